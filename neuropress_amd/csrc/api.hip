// Library-level entry points: version, thread-local error text, launch check.
#include <stdarg.h>
#include <stdio.h>

#include <stdlib.h>

#include "../../include/npamd_diag.h"
#include "gemm_tile2.hpp"
#include "gemv.hpp"

namespace npamd {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

hipError_t& launch_status() {
  thread_local hipError_t status = hipSuccess;
  return status;
}

int check_launch(const char* what) {
  const hipError_t e = launch_status();
  if (e == hipSuccess) return NPAMD_OK;
  launch_status() = hipSuccess;
  (void)hipGetLastError();  // reported here: not the next call's
  return fail(NPAMD_ERR_LAUNCH, "%s: launch failed: %s", what, hipGetErrorString(e));
}

const char* error_text() { return g_err; }

static int env_int(const char* name, int dflt) {
  const char* v = getenv(name);
  return (v && *v) ? atoi(v) : dflt;
}

// The NPAMD_* tuning variables, read once per process (initialisation of a function-local
// static is thread-safe); launches only read the table.  npamd_diag_reload_tuning() reads them
// again, for tests and tuning runs that change them between launches.
static Tuning read_tuning() {
  Tuning t;
  t.gemv_lds_cb = env_int("NPAMD_GEMV_LDS_CB", 1);
  t.tile_lds_cb = env_int("NPAMD_TILE_LDS_CB", 1);
  t.gemv_lds_x = env_int("NPAMD_GEMV_LDS_X", 0);
  t.gemv_r = env_int("NPAMD_GEMV_R", 0);
  t.gemv_spw = env_int("NPAMD_GEMV_SPW", 0);
  t.gemv_parts = env_int("NPAMD_GEMV_PARTS", 0);
  t.gemv_xstage = env_int("NPAMD_GEMV_XSTAGE", 1);
  t.tile_splits = env_int("NPAMD_TILE_SPLITS", 0);
  t.tile_mw = env_int("NPAMD_TILE_MW", 0);
  t.tile_wide = env_int("NPAMD_TILE_WIDE", 1);
  t.tile_call = env_int("NPAMD_TILE_CALL", 0);
  t.tile_spins = env_int("NPAMD_TILE_SPINS", 0);
  t.slice_tiles = env_int("NPAMD_SLICE_TILES", 0);
  t.slice_parts = env_int("NPAMD_SLICE_PARTS", 0);
  t.q4_rows = env_int("NPAMD_Q4_ROWS", 0);
  t.q4_rowwise = env_int("NPAMD_Q4_ROWWISE", 1);
  t.q4_rowwise_bf16 = env_int("NPAMD_Q4_ROWWISE_BF16", 0);
  t.q4_stream = env_int("NPAMD_Q4_STREAM", 1);
  t.dense_tile = env_int("NPAMD_DENSE_TILE", 0);
  t.dense_splits = env_int("NPAMD_DENSE_SPLITS", 0);
  t.table_tile = env_int("NPAMD_TABLE_TILE", 0);
  return t;
}

static Tuning& tuning_table() {
  static Tuning table = read_tuning();
  return table;
}

const Tuning& tuning() { return tuning_table(); }

static int device_cu_count() {
  // Looked up at most a few times per process (racing first callers all store the same value).
  static std::atomic<int> cached{0};
  int cus = cached.load(std::memory_order_relaxed);
  if (cus == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      cus = prop.multiProcessorCount;
    if (cus <= 0) cus = 256;
    cached.store(cus, std::memory_order_relaxed);
  }
  return cus;
}

// One "job" = one 16-row tile x one 256-k step.  The kernel lasts about one
// HBM round trip, so the plan aims at every job's packed bytes being requested
// as soon as the grid starts: jobs per wave is kept near jobs / (16 waves * CUs).
// NPAMD_GEMV_R / NPAMD_GEMV_SPW override the choice (tuning aid).
bool gemv_lds_codebook_enabled() { return tuning().gemv_lds_cb != 0; }
bool tile_lds_codebook_enabled() { return tuning().tile_lds_cb != 0; }
bool gemv_lds_activations_forced() { return tuning().gemv_lds_x != 0; }
// One row tile per block, us, straight from memory / staged, 65536-row codebook 4096 x 14336 35.8 / 34.6 at 4 tokens,
// 37.8 / 35.4 at 8, 42.4 / 37.6 at 16, 52 / 41 at 32; 4096 rows, looked up in LDS, 11.2 / 9.2 at 4, 13.2 / 10.2 at 8,
// 19.1 / 12.7 at 16.  With more row tiles per block: see launch_fused_gemv.
int& last_gemv_staged() {
  static thread_local int staged = -1;
  return staged;
}

bool gemv_stage_activations(int M) {
  const int mode = tuning().gemv_xstage;
  return mode >= 2 || (mode == 1 && M >= 3);
}

// Whether the blocks of 17 and more tokens look a table that LDS could hold up in memory: where their lookups are few, the copy
// is what a block waits for, and a table of more than 32 KiB next to 16 KiB of activations per wave leaves room for six waves.
// fp16, 64 tokens, table in LDS / in memory, us: 256 rows 512 x 512 4.7 / 4.0, 8192 x 512 6.4 / 6.0, 1024 x 1024 4.8 / 4.7, but at 512
// tokens 1024 x 1024 (8192 lookups per compute unit) 6.9 / 9.2 and 2048 x 2048 (whose blocks have 4096) 5.7 / 5.7; 4096 rows 512 x 2048
// 7.3 / 5.4, 2048 x 2048 10.0 / 7.0, 1024 x 4096 9.6 / 8.1, at 128 tokens 9.1 / 12.5 and 9.8 / 10.3.
bool gemv_wide_looks_up_in_memory(int M, int row_tiles, int chunks, int cb_bytes) {
  const int cus = device_cu_count();
  const int64_t block = (int64_t)16 * chunks * 8, fullest = (row_tiles + cus - 1) / cus * block;
  return fullest <= 4096 && (block <= 2048 || (cb_bytes > 32 * 1024 && M > 24));
}

// Row tiles of a block with staged activations next to the table: two where one leaves compute units a second round of blocks
// (us with one / two / four, 24 tokens: 14336 x 4096 21.6 / 13.7 / 15.6 with 256 rows, 23.4 / 14.7 / 16.0 with 4096; 128 tokens: 2048 x
// 2048 9.7 / 6.5 / 11.1, 4096 x 1024 9.5 / 6.9 / 9.8; 256 tokens 1024 x 4096 13.1 / 8.4 / 16.5).  Large tables past 24 tokens leave room for
// six waves: four row tiles, activations from memory, on large grids (14336 x 4096 at 32 tokens 32.9 / 20.4 / 18.4).
int gemv_wide_row_tiles(int M, int row_tiles, int cb_bytes) {
  const int cus = device_cu_count();
  if (cb_bytes > 32 * 1024 && M > 24 && row_tiles * 10 >= cus * 24) return 4;
  return row_tiles > cus ? 2 : 1;
}

GemvPlan plan_gemv(int N, int chunks, int max_r, int max_waves_cap, bool exact) {
  const int steps = (chunks + 3) / 4;
  const int tiles = (N + 15) / 16;
  const int64_t jobs = (int64_t)tiles * steps;
  const int cus = device_cu_count();
  const int64_t target_waves = (int64_t)cus * 16;
  int jpw = (int)((jobs + target_waves - 1) / target_waves);
  if (jpw < 1) jpw = 1;
  GemvPlan p;
  // Row tiles of one block share the x operands (every block reads all of x, from L2: with R
  // tiles per block that traffic, which passes the weight bytes at a few tokens, drops R-fold)
  // and one copy of the codebook in LDS.  The largest R that leaves blocks for at least 0.6 of
  // the compute units wins at every token count, measured on N = 2048 ... 28672.
  p.R = (tiles * 10 >= cus * 24) ? 4 : (tiles * 10 >= cus * 12) ? 2 : 1;
  if (p.R > max_r || exact) p.R = max_r;
  int spw = (jpw + p.R - 1) / p.R;
  const int r_env = tuning().gemv_r;
  if (r_env == 1 || r_env == 2 || r_env == 4) p.R = r_env;
  const int spw_env = tuning().gemv_spw;
  if (spw_env > 0) spw = spw_env;
  int max_waves = p.R >= 4 ? 8 : 16;
  if (max_waves > max_waves_cap) max_waves = max_waves_cap;
  if ((steps + spw - 1) / spw > max_waves) spw = (steps + max_waves - 1) / max_waves;
  p.steps_per_wave = spw;
  p.waves = (steps + spw - 1) / spw;
  return p;
}

// Measured, one token, 16 rows per block against 8 / 4 (us): residual VQ 1024 x 4096 7.7 -> 4.4,
// 65536-row codebook 1024 x 4096 8.4 -> 4.8, 2048 x 4096 9.2 -> 7.1 and 1024 x 1024 3.8 -> 3.3,
// int4 1024 x 4096 at two tokens 5.8 -> 3.8, 2048 x 8192 with a 4096-row table in LDS 6.5 -> 5.5,
// 2048 x 4096 with it 5.0 -> 4.5; but 2048 x 2048 and 512 x 2048 with that table 4.2 -> 4.4 and
// 4.15 -> 4.9 (every block copies the 64 KiB first, and there are then two or four times as
// many), 4096 x 4096 (whole tiles cover the compute units) 5.3 -> 5.5.  Hence: K of at least 512
// per part, whole tiles leave a quarter of the compute units empty, and a block keeps at least
// one lookup per row of the table it copies.
int plan_gemv_parts(int M, int N, int chunks, int lds_rows) {
  const int env = tuning().gemv_parts;
  const int cus = device_cu_count();
  int h = 1;
  while (h < 4) {
    const int next = 2 * h;
    const int tiles = (N + 16 / h - 1) / (16 / h);
    const bool fits = M <= 16 / next && chunks >= 8 * next;
    const bool wanted = tiles * 4 < cus * 3;
    const bool pays = (int64_t)(16 / next) * chunks * 8 >= (int64_t)lds_rows;
    if (!(fits && wanted && pays)) break;
    h = next;
  }
  if (env == 1 || env == 2 || env == 4) h = (M <= 16 / env) ? env : 1;
  return h;
}

GemvPlan plan_gemv_rows(int N, int rows, int steps) {
  const int tiles = (N + rows - 1) / rows;
  const int64_t jobs = (int64_t)tiles * steps;
  const int64_t target_waves = (int64_t)device_cu_count() * 16;
  int spw = (int)((jobs + target_waves - 1) / target_waves);
  if (spw < 1) spw = 1;
  if ((steps + spw - 1) / spw > 16) spw = (steps + 15) / 16;
  GemvPlan p;
  p.R = 1;
  p.steps_per_wave = spw;
  p.waves = (steps + spw - 1) / spw;
  return p;
}

bool gemv_perm_keeps_occupancy(int M, int N, int chunks, int cb_bytes) {
  const int cbl = (cb_bytes > 0 && cb_bytes <= kGemvLdsCodebookMax && gemv_lds_codebook_enabled()) ? cb_bytes : 0;
  const GemvPlan plan = plan_gemv(N, chunks, cbl ? 4 : 2);
  const int red = ((plan.waves * M * 16 * plan.R + 3) & ~3) * (int)sizeof(float);
  const int xb = M * chunks * 64 * 2;
  const int lds = red + (cbl > xb ? cbl : xb) + xb;
  const int blocks = (N + 16 * plan.R - 1) / (16 * plan.R);
  return lds <= 80 * 1024 || (blocks <= device_cu_count() && lds <= 160 * 1024);
}

int plan_tile_splits(int M, int N, int chunks, int mw) {
  const int env = tuning().tile_splits;
  const int cus = device_cu_count();
  const int blocks = ((N + 63) / 64) * ((M + 128 * mw - 1) / (128 * mw));
  int splits = 1;
  if (env > 0) splits = env;
  else if (blocks * 10 < cus * 7) splits = cus / blocks;
  const int max_by_k = chunks / 8 > 1 ? chunks / 8 : 1;
  if (splits > max_by_k) splits = max_by_k;
  if (splits > 16) splits = 16;
  return splits < 1 ? 1 : splits;
}

int tile2_mode() { return tuning().tile_wide; }

int plan_tile2_splits(int M, int N, int chunks, int mw) {
  const int env = tuning().tile_splits;
  const int cus = device_cu_count();
  const int blocks = ((N + kT2Cols - 1) / kT2Cols) * ((M + 128 * mw - 1) / (128 * mw));
  int splits = 1;
  if (env > 0) splits = env;
  else if (blocks * 10 < cus * 7) splits = cus / blocks;
  const int max_by_k = chunks / 8 > 1 ? chunks / 8 : 1;
  if (splits > max_by_k) splits = max_by_k;
  if (splits > 16) splits = 16;
  return splits < 1 ? 1 : splits;
}

extern "C" int64_t npamd_gemm_tile_workspace_bytes(int M, int N, int K);

int plan_tile_mw(int M) {
  const int mw_env = tuning().tile_mw;
  if (mw_env >= 1 && mw_env <= 3) return mw_env;
  const int mw = (M + 127) / 128;
  return mw < 1 ? 1 : (mw > 3 ? 3 : mw);
}

}  // namespace npamd

extern "C" int npamd_version(void) { return 3; }

extern "C" int npamd_gemv_stages_activations(int M, int N, int K, int nc) {
  if (M < 1 || M > NPAMD_GEMV_MAX_M || N < 1 || K < 64 || K % 64 || nc < 0) return 0;
  return nc ? npamd::vq_gemv_plan_stages(M, N, K, nc) : npamd::q_gemv_plan_stages(M, N, K);
}

// Next to a table in LDS staging keeps the GEMV ahead at 17 and 24 tokens, not to 32: 4096 x 14336 with 4096 rows 15.4 / 17.8 / 24.3 us against
// 21.6 / 21.8 / 21.9 of the tile GEMM, 2048 x 14336 at 24 16.0 against 16.8; the blocks entries' line (npamd_gemv_blocks_preferred) tells them apart.
extern "C" int npamd_gemv_ahead_of_tile(int M, int N, int K, int nc) {
  const bool table_in_lds = M > 16 && nc > 0 && nc <= npamd::kGemvLdsCodebookMax / 16;
  return table_in_lds ? 0 : npamd_gemv_stages_activations(M, N, K, nc);
}

extern "C" int npamd_diag_last_gemv_staged(void) { return npamd::last_gemv_staged(); }

extern "C" void npamd_diag_reload_tuning(void) { npamd::tuning_table() = npamd::read_tuning(); }

extern "C" int64_t npamd_gemm_tile_workspace_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K < 64) return 0;
  const int mw = npamd::plan_tile_mw(M);
  const int splits = npamd::plan_tile_splits(M, N, K / 64, mw);
  const int64_t narrow = splits > 1 ? (int64_t)splits * M * N * 4 : 0;
  int64_t wide = 0;
  if (npamd::tile2_mode()) {
    wide = npamd::tile2_workspace_bytes(M, N, K / 64, mw);
    const int64_t wide_q = npamd::tile2_workspace_bytes(M, N, K / 64, npamd::plan_tile2_q_mw(M));
    if (wide_q > wide) wide = wide_q;
  }
  return narrow > wide ? narrow : wide;
}

extern "C" const char* npamd_last_error(void) { return npamd::error_text(); }
