#include "rules.h"

#include <array>
#include <cmath>
#include <cstring>

#include "../kernels/iu8_pf_law.h"
#include "abi.h"
#include "util.h"

namespace iu8 {

static const DecVariant DEC_VARIANTS[] = {
#define IU8_DEC_VARIANT(name, TM, W8, NT, KW, WPB, D, ALDS, ACC) {#name, TM, W8, NT, KW, WPB, D, ALDS, ACC},
#define IU8_DEC_TAP(name, TM, W8, NT, KW, WPB, D, ALDS, ACC) {#name, TM, W8, NT, KW, WPB, D, ALDS, ACC},
#include "../kernels/iu8_variants.def"
};
static const PfVariant PF_VARIANTS[] = {
#define IU8_PF_VARIANT(name, W8, WMW, WNW, TM, TN, ACC, ST, OCC, DEEP, KW) {#name, W8, WMW, WNW, TM, TN, ACC, OCC, KW},
#define IU8_PF_TAP(name, W8, WMW, WNW, TM, TN, ACC, ST, OCC, DEEP, KW) {#name, W8, WMW, WNW, TM, TN, ACC, OCC, KW},
#include "../kernels/iu8_variants.def"
};
static const WideVariant WIDE_VARIANTS[] = {
#define IU8_WIDE_VARIANT(name, TM, W8, NT, KW, D) {#name, TM, W8, NT, KW},
#include "../kernels/iu8_variants.def"
};
static const RowsVariant ROWS_VARIANTS[] = {
#define IU8_ROWS_VARIANT(name, TM, W8, NT, KW, D) {#name, TM, W8, NT, KW},
#include "../kernels/iu8_variants.def"
};
static const DecVariant PAIR_VARIANTS[] = {
#define IU8_PAIR_VARIANT(name, TM, NT, KW, WPB, D, ALDS, BFIRST) {#name, TM, false, NT, KW, WPB, D, ALDS, false},
#include "../kernels/iu8_variants.def"
};

const DecVariant *dec_variant(const std::string &name) {
  for (const DecVariant &v : DEC_VARIANTS)
    if (name == v.name) return &v;
  return nullptr;
}
const DecVariant *pair_variant(const std::string &name) {
  for (const DecVariant &v : PAIR_VARIANTS)
    if (name == v.name) return &v;
  return nullptr;
}
const WideVariant *wide_variant(const std::string &name) {
  for (const WideVariant &v : WIDE_VARIANTS)
    if (name == v.name) return &v;
  return nullptr;
}
const RowsVariant *rows_variant(const std::string &name) {
  for (const RowsVariant &v : ROWS_VARIANTS)
    if (name == v.name) return &v;
  return nullptr;
}
const PfVariant *pf_variant(const std::string &name) {
  for (const PfVariant &v : PF_VARIANTS)
    if (name == v.name) return &v;
  return nullptr;
}

int fill_slots(const std::string &kernel, saber_iu8_desc *d) {
  const Signature *sig = signature_for(kernel);
  if (!sig) return fail(SABER_IU8_E_RULE, kernel + ": no declared signature");
  if (sig->size() > sizeof(d->args) / sizeof(d->args[0])) return fail(SABER_IU8_E_RULE, kernel + ": too many arguments");
  d->n_args = (uint32_t)sig->size();
  uint32_t off = 0;
  for (size_t i = 0; i < sig->size(); ++i) {
    saber_iu8_slot &s = d->args[i];
    memset(&s, 0, sizeof s);
    copy_name(s.name, sizeof s.name, (*sig)[i].name);
    s.offset = off = pack_at((*sig)[i], off);
    s.size = (*sig)[i].size();
    off += s.size;
    s.kind = (*sig)[i].kind == ArgKind::Buffer ? SABER_IU8_ARG_BUFFER
             : (*sig)[i].kind == ArgKind::F32  ? SABER_IU8_ARG_F32
             : (*sig)[i].kind == ArgKind::I64  ? SABER_IU8_ARG_I64
                                               : SABER_IU8_ARG_I32;
  }
  d->kernarg_bytes = off;
  return 0;
}

void set_i32(saber_iu8_desc *d, const char *name, int64_t v) {
  for (uint32_t i = 0; i < d->n_args; ++i)
    if (!strcmp(d->args[i].name, name)) {
      d->args[i].kind = d->args[i].size == 8 ? SABER_IU8_ARG_I64 : SABER_IU8_ARG_I32;
      d->args[i].ival = v;
    }
}
void set_buffer(saber_iu8_desc *d, const char *name) {
  for (uint32_t i = 0; i < d->n_args; ++i)
    if (!strcmp(d->args[i].name, name)) d->args[i].kind = SABER_IU8_ARG_BUFFER;
}
void set_null(saber_iu8_desc *d, const char *name) {
  for (uint32_t i = 0; i < d->n_args; ++i)
    if (!strcmp(d->args[i].name, name)) d->args[i].kind = SABER_IU8_ARG_NULL_BUFFER;
}

static void add_ws(saber_iu8_desc *d, const char *name, uint32_t kind, uint64_t bytes, uint32_t zero_once) {
  saber_iu8_workspace &w = d->workspaces[d->n_workspaces++];
  memset(&w, 0, sizeof w);
  copy_name(w.name, sizeof w.name, name);
  w.kind = kind;
  w.bytes = bytes;
  w.zero_once = zero_once;
}

static int check_shape(const char *op, uint32_t m, uint32_t n, uint32_t k) {
  // the reference's refusals (macaq_iu8.rs:288-297), by name
  if (m == 0 || n == 0 || k == 0)
    return fail(SABER_IU8_E_RULE, fmt("%s: %u x %u x %u has nothing to do; an empty launch is a caller bug", op, m, n, k));
  if (n % 16 != 0 || k % 128 != 0)
    return fail(SABER_IU8_E_RULE,
                fmt("%s: N=%u must be a multiple of 16 (whole fragments) and K=%u of 128 (the slab)", op, n, k));
  // the kernels take their sizes as int; and a count of blocks or tiles, (size + block - 1) / block in 32 bits, wraps to none
  if (m > INT32_MAX || n > INT32_MAX || k > INT32_MAX)
    return fail(SABER_IU8_E_RULE, fmt("%s: %u x %u x %u is past the kernels' 32-bit sizes", op, m, n, k));
  return 0;
}

static int describe_dec(const DecVariant &v, uint32_t m, uint32_t n, uint32_t k, uint32_t ks, saber_iu8_desc *d) {
  const char *op = v.w8 ? "gemm_i8a8" : "gemm_i4a8";
  if (int rc = check_shape(op, m, n, k)) return rc;
  if (m > (uint32_t)v.tm * 16) return fail(SABER_IU8_E_RULE, fmt("%s: %s holds %d rows, M=%u", op, v.name, v.tm * 16, m));
  if (ks == 0 || ks > k / 128) return fail(SABER_IU8_E_RULE, fmt("%s: split %u of %u K steps", op, ks, k / 128));
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8");
  copy_name(d->kernel, sizeof d->kernel, v.name);
  const uint32_t bn = v.block_n(m, n, k, ks), nblk = (n + bn - 1) / bn;
  d->grid[0] = nblk, d->grid[1] = 1, d->grid[2] = ks;
  d->block[0] = v.threads(), d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = ks;
  if (int rc = fill_slots(v.name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", n);
  set_i32(d, "k", k);
  if (ks == 1) {
    // named-null at ks 1: the kernel must not dereference them (macaq_iu8.rs:447-451)
    set_null(d, "decode_partial");
    set_null(d, "decode_counter");
  } else {
    add_ws(d, "decode_partial", SABER_IU8_WS_SCRATCH, (uint64_t)ks * m * n * 4, 0);
    add_ws(d, "decode_counter", SABER_IU8_WS_PERSISTENT, (uint64_t)nblk * 4, 1);
  }
  return 0;
}

// The tile GEMM addresses its operands with 32-bit byte offsets from a per-step base.
static uint64_t a_operand_bytes(uint32_t m, uint32_t k) { return (uint64_t)((m + 15) / 16 * 16) * k; }
static uint64_t w_operand_bytes(bool w8, uint32_t n, uint32_t k) { return (uint64_t)n * k / (w8 ? 1 : 2); }
static bool tile_operands_hold(bool w8, uint32_t m, uint32_t n, uint32_t k) {
  return a_operand_bytes(m, k) <= 0xFFFFFFFFull && w_operand_bytes(w8, n, k) <= 0xFFFFFFFFull;
}

// `ks` > 0 names the cell's split form (`<cell>_ks`, the decode kernarg list): gridDim.z shares of the
// K steps, none of them empty, `grid[0]` persistent workgroups a share.
static int describe_pf(const PfVariant &v, uint32_t m, uint32_t n, uint32_t k, uint32_t ks, saber_iu8_desc *d) {
  const char *op = v.w8 ? "gemm_i8a8" : "gemm_i4a8";
  if (int rc = check_shape(op, m, n, k)) return rc;
  if (!tile_operands_hold(v.w8, m, n, k))
    return fail(SABER_IU8_E_RULE, fmt("%s: %u x %u x %u puts an operand past 4 GiB (A %llu B, W %llu B), more than the tile GEMM addresses",
                                      op, m, n, k, (unsigned long long)a_operand_bytes(m, k), (unsigned long long)w_operand_bytes(v.w8, n, k)));
  const std::string name = std::string(v.name) + (ks ? "_ks" : "");
  if (ks) {
    const uint32_t steps = k / 128, spb = (steps + ks - 1) / ks;
    if (ks > steps || (uint64_t)spb * (ks - 1) >= steps)
      return fail(SABER_IU8_E_RULE, fmt("%s: %u shares of %u K steps would leave one empty", op, ks, steps));
  }
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8");
  copy_name(d->kernel, sizeof d->kernel, name);
  const uint32_t gx = (n + v.block_n() - 1) / v.block_n(), gy = (m + v.block_m() - 1) / v.block_m();
  // persistent: OCC workgroups a CU walk the tiles (the kernel derives gx, gy from m, n)
  const uint64_t tiles = (uint64_t)gx * gy, slots = std::max<uint64_t>(1, (uint64_t)CU_COUNT * v.occ / std::max(ks, 1u));
  d->grid[0] = (uint32_t)(tiles < slots ? tiles : slots), d->grid[1] = 1, d->grid[2] = std::max(ks, 1u);
  d->block[0] = v.threads(), d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = std::max(ks, 1u);
  if (int rc = fill_slots(name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", n);
  set_i32(d, "k", k);
  if (ks == 1) {
    set_null(d, "decode_partial");
    set_null(d, "decode_counter");
  } else if (ks > 1) {
    add_ws(d, "decode_partial", SABER_IU8_WS_SCRATCH, (uint64_t)ks * m * n * 4, 0);
    add_ws(d, "decode_counter", SABER_IU8_WS_PERSISTENT, tiles * 4, 1);
  }
  return 0;
}

static int describe_wide(const WideVariant &v, uint32_t m, uint32_t n, uint32_t k, saber_iu8_desc *d) {
  const char *op = v.w8 ? "gemm_i8a8" : "gemm_i4a8";
  if (int rc = check_shape(op, m, n, k)) return rc;
  if (m > (uint32_t)v.block_m()) return fail(SABER_IU8_E_RULE, fmt("%s: %s holds %d rows, M=%u", op, v.name, v.block_m(), m));
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8");
  copy_name(d->kernel, sizeof d->kernel, v.name);
  d->grid[0] = (n + v.block_n() - 1) / v.block_n(), d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = v.threads(), d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(v.name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", n);
  set_i32(d, "k", k);
  return 0;
}

// Blocks in whole eighths: the kernel gives an XCD a run of them, column blocks of one row tile side by side.
static int describe_rows_cell(const RowsVariant &v, uint32_t m, uint32_t n, uint32_t k, saber_iu8_desc *d) {
  const char *op = v.w8 ? "gemm_i8a8" : "gemm_i4a8";
  if (int rc = check_shape(op, m, n, k)) return rc;
  const uint64_t blocks = (uint64_t)((n + v.block_n() - 1) / v.block_n()) * ((m + v.block_m() - 1) / v.block_m());
  if (blocks > ROWS_CELL_BLOCKS_MAX || (uint64_t)v.block_m() * k > INT32_MAX)
    return fail(SABER_IU8_E_RULE, fmt("%s: %s holds %u blocks of rows under 2 GiB, %u x %u x %u", op, v.name, ROWS_CELL_BLOCKS_MAX, m, n, k));
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8");
  copy_name(d->kernel, sizeof d->kernel, v.name);
  d->grid[0] = (uint32_t)((blocks + 7) / 8 * 8), d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = v.threads(), d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(v.name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", n);
  set_i32(d, "k", k);
  return 0;
}

static uint64_t staged_bytes(uint32_t m, uint32_t k);
// The streaming decode cell of M rows: tm 16-row tiles; one tile's live rows staged in LDS when they fit the 20 KiB
// form, else streamed from L2 beside the weights.
static std::string dec_stream_name(const char *tag, uint32_t m, uint32_t k) {
  const uint32_t tm = (m + 15) / 16;
  std::string name = fmt("macaq_iu8_dec_%s_tm%u", tag, tm);
  if (tm == 1) {
    uint32_t mr = 1;
    while (mr < m) mr *= 2;
    if ((uint64_t)mr * k > 20 * 1024) name += "_a0";
  }
  return name;
}

// The persistent GEMV of up to 16 quantised rows whose 16-row tile is staged once a workgroup in 80 KiB of LDS
// (`macaq_iu8_dec_{w4,w8}_tm1_s80`): the fused forms' geometry (16 waves, 32 columns a block, at most 8 blocks a
// workgroup) on the decode kernarg list.
bool staged80_holds(uint32_t m, uint32_t k) { return m >= 1 && m <= 16 && staged_bytes(m, k) <= 80 * 1024; }
static bool staged80_tile_holds(uint32_t m, uint32_t k) { return m >= 1 && m <= 16 && (uint64_t)k * 16 <= 80 * 1024; }
// `rows_form`: the kernel that takes the live rows' pieces of the tile (`_s80r`: few rows of a long K); else the
// whole-tile kernel (`_s80`, K <= 5120 at any row count)
static int describe_s80(bool w8, bool rows_form, uint32_t m, uint32_t n, uint32_t k, uint32_t ks, saber_iu8_desc *d) {
  const char *op = w8 ? "gemm_i8a8" : "gemm_i4a8";
  const std::string name = fmt("macaq_iu8_dec_%s_tm1_s80%s", w8 ? "w8" : "w4", rows_form ? "r" : "");
  if (int rc = check_shape(op, m, n, k)) return rc;
  if (ks != 1) return fail(SABER_IU8_E_RULE, name + ": the staged form does not split K");
  if (rows_form ? !staged80_holds(m, k) : !staged80_tile_holds(m, k))
    return fail(SABER_IU8_E_RULE, rows_form ? fmt("%s: %u rows (rounded up to a power of two) of %u do not fit 80 KiB", name.c_str(), m, k)
                                            : fmt("%s: %u rows of %u do not fit one 16-row tile in 80 KiB (K <= 5120)", name.c_str(), m, k));
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8");
  copy_name(d->kernel, sizeof d->kernel, name);
  d->grid[0] = fused_grid((n + 31) / 32), d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = 1024, d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", n);
  set_i32(d, "k", k);
  set_null(d, "decode_partial");
  set_null(d, "decode_counter");
  return 0;
}

int describe(const std::string &kernel, uint32_t m, uint32_t n, uint32_t k, uint32_t ks, saber_iu8_desc *out) {
  if (kernel == "macaq_iu8_dec_w4_tm1_s80" || kernel == "macaq_iu8_dec_w8_tm1_s80") return describe_s80(kernel[15] == '8', false, m, n, k, ks, out);
  if (kernel == "macaq_iu8_dec_w4_tm1_s80r" || kernel == "macaq_iu8_dec_w8_tm1_s80r") return describe_s80(kernel[15] == '8', true, m, n, k, ks, out);
  if (const DecVariant *v = dec_variant(kernel)) return describe_dec(*v, m, n, k, ks, out);
  if (const WideVariant *v = wide_variant(kernel)) {
    if (ks != 1) return fail(SABER_IU8_E_RULE, kernel + ": the wide streamed cell does not split K");
    return describe_wide(*v, m, n, k, out);
  }
  if (const RowsVariant *v = rows_variant(kernel)) {
    if (ks != 1) return fail(SABER_IU8_E_RULE, kernel + ": the streamed cell on row tiles does not split K");
    return describe_rows_cell(*v, m, n, k, out);
  }
  if (const PfVariant *v = pf_variant(kernel)) {
    if (ks != 1) return fail(SABER_IU8_E_RULE, kernel + ": the prefill tile does not split K (its `_ks` form does)");
    return describe_pf(*v, m, n, k, 0, out);
  }
  if (kernel.size() > 3 && kernel.compare(kernel.size() - 3, 3, "_ks") == 0)
    if (const PfVariant *v = pf_variant(kernel.substr(0, kernel.size() - 3))) {
      if (!signature_for(kernel)) return fail(SABER_IU8_E_RULE, kernel + ": no such split form");
      return describe_pf(*v, m, n, k, ks, out);
    }
  // the tile GEMM with the quantisation fused into its A-tile load: the geometry of the cell it names
  if (kernel.rfind("macaq_iu8_pfq_", 0) == 0)
    if (const PfVariant *v = pf_variant("macaq_iu8_pf_" + kernel.substr(14))) {
      // the cells that have a fused-quant form (registers for the bf16 pieces in flight, whole A fragments a wave)
      static const char *const PFQ[] = {"w4_t128x128", "w8_t128x128", "w4_t128x128_o2", "w4_t256x160", "w8_t256x160"};
      bool has = false;
      for (const char *c : PFQ) has = has || kernel.substr(14) == c;
      if (!has || ks != 1) return fail(SABER_IU8_E_RULE, kernel + ": no such fused-quant form");
      if ((uint64_t)m * k * 2 > 0xFFFFFFFFull) return fail(SABER_IU8_E_RULE, fmt("%s: %u rows of %u bf16 pass 4 GiB", kernel.c_str(), m, k));
      if (int rc = describe_pf(*v, m, n, k, 0, out)) return rc;
      copy_name(out->kernel, sizeof out->kernel, kernel);
      copy_name(out->op, sizeof out->op, v->w8 ? "linear_i8a8_pfq" : "linear_i4a8_pfq");
      if (int rc = fill_slots(kernel, out)) return rc;
      set_i32(out, "m", m), set_i32(out, "n", n), set_i32(out, "k", k);
      return 0;
    }
  // a name of the reference's symbol set that this object does not carry (gfx1201 tile shapes): the
  // request is for the op at this shape, and the gfx950 law picks the cell
  int w8 = 0;
  const char *note = "";
  const int r = ref_symbol_by_law(kernel, &w8, &note);
  if (r > 0) {
    if (ks != 1) return fail(SABER_IU8_E_RULE, kernel + ": answered by the launch law, which picks the split itself");
    return resolve(w8 ? SABER_IU8_W8 : SABER_IU8_W4, m, n, k, out);
  }
  if (r < 0) return fail(SABER_IU8_E_RULE, kernel + ": " + note);
  return fail(SABER_IU8_E_RULE, kernel + ": not a kernel of the macaq_iu8 object");
}

static bool int_arg(const saber_iu8_desc &d, const char *name, int64_t *v) {
  for (uint32_t i = 0; i < d.n_args; ++i)
    if (!strcmp(d.args[i].name, name) && (d.args[i].kind == SABER_IU8_ARG_I32 || d.args[i].kind == SABER_IU8_ARG_I64)) {
      *v = d.args[i].ival;
      return true;
    }
  return false;
}

// The decode pair: each half is exactly the descriptor `resolve` / `describe` gave it alone (its
// split count, its partial slab and counters), the two grids end to end, problem 0 first
// (macaq_iu8.rs:632-704). Refused unless both halves are W4 decode cells of one kernel (so one row
// tiling and one staging form), M and K.
int pair(const saber_iu8_desc &first, const saber_iu8_desc &second, saber_iu8_desc *out, int order) {
  static const char PREFIX[] = "macaq_iu8_dec_w4_";
  // a half the law gave the staged persistent form, or 17 to 48 rows at another block width, is paired as its streamed
  // form, which is the pair kernels' geometry, on the split count it was given
  // (and up to 48 rows the streamed cell on row tiles)
  auto other_form = [](const saber_iu8_desc &h) {
    int64_t hm = 0;
    if (const RowsVariant *v = rows_variant(h.kernel)) return !v->w8 && int_arg(h, "m", &hm) && hm <= ROWS_CELL_FEW_ROWS;
    return !strncmp(h.kernel, "macaq_iu8_dec_w4_tm1_s80", 24) || !strcmp(h.kernel, "macaq_iu8_dec_w4_tm2_n1") ||
           !strcmp(h.kernel, "macaq_iu8_dec_w4_tm3_n2");
  };
  for (const saber_iu8_desc *h : {&first, &second})
    if (other_form(*h)) {
      saber_iu8_desc s[2];
      const saber_iu8_desc *in[2] = {&first, &second};
      for (int i = 0; i < 2; ++i) {
        int64_t hm = 0, hn = 0, hk = 0;
        s[i] = *in[i];
        if (other_form(*in[i])) {
          if (!int_arg(*in[i], "m", &hm) || !int_arg(*in[i], "n", &hn) || !int_arg(*in[i], "k", &hk))
            return fail(SABER_IU8_E_RULE, "macaq iu8 pair: a half without its m, n, k");
          if (int rc = describe(dec_stream_name("w4", (uint32_t)hm, (uint32_t)hk), (uint32_t)hm, (uint32_t)hn, (uint32_t)hk, in[i]->ks, &s[i])) return rc;
        }
      }
      return pair(s[0], s[1], out, order);
    }
  const std::string k0 = first.kernel, k1 = second.kernel;
  const DecVariant *v0 = dec_variant(k0), *v1 = dec_variant(k1);
  int64_t m0 = 0, kk0 = 0, n0 = 0, m1 = 0, kk1 = 0, n1 = 0;
  const bool ints = int_arg(first, "m", &m0) && int_arg(first, "k", &kk0) && int_arg(first, "n", &n0) &&
                    int_arg(second, "m", &m1) && int_arg(second, "k", &kk1) && int_arg(second, "n", &n1);
  if (!v0 || !v1 || !ints || v0->w8 || v1->w8 || v0->acc || v1->acc || k0 != k1 || m0 != m1 || kk0 != kk1)
    return fail(SABER_IU8_E_RULE, fmt("macaq iu8 pair: halves `%s` M %lld K %lld and `%s` M %lld K %lld are not two W4 cells of one M, K",
                                      k0.c_str(), (long long)m0, (long long)kk0, k1.c_str(), (long long)m1, (long long)kk1));
  // The block order by tm (speed data; both orders give the same bytes): the second problem's
  // workgroups first (`pairb`), as the reference's PAIR_BA_FIRST has it at every tm
  // (macaq_iu8.rs:549-553) -- the small half then does not sit in the launch's tail.
  static const bool PAIR_B_FIRST[4] = {true, true, true, true};
  const bool b_first = order < 0 ? PAIR_B_FIRST[std::min(std::max(v0->tm, 1), 4) - 1] : order > 0;
  const char *form = b_first ? "pairb" : "pair";
  const std::string name = std::string("macaq_iu8f_") + form + "_w4_" + k0.substr(sizeof PREFIX - 1);
  const DecVariant *pv = pair_variant(name);
  if (!pv) return fail(SABER_IU8_E_RULE, name + ": the fused object carries no such pair");
  const uint32_t ks0 = first.ks, ks1 = second.ks;
  // A half's block width is its own launch's. Two unsplit halves that would both take 64-column blocks share the CUs, so their
  // columns together say whether those pay: 9600 + 9600 x 8192 at 5 / 16 rows on 64 columns 18.2 / 19.0 us, on 32 15.5 / 17.3.
  auto width = [&](int64_t n, uint32_t ks) { return pv->block_n((uint32_t)m0, (uint32_t)n, (uint32_t)kk0, ks); };
  int bn0 = width(n0, ks0), bn1 = width(n1, ks1);
  if (ks0 == 1 && ks1 == 1 && bn0 != pv->own_n() && bn1 != pv->own_n()) bn0 = bn1 = width(n0 + n1, 1);
  const uint32_t nb0 = (uint32_t)((n0 + bn0 - 1) / bn0), nb1 = (uint32_t)((n1 + bn1 - 1) / bn1);
  memset(out, 0, sizeof *out);
  copy_name(out->op, sizeof out->op, "gemm_i4a8_pair");
  copy_name(out->plugin, sizeof out->plugin, "macaq_iu8f");
  copy_name(out->kernel, sizeof out->kernel, name);
  out->grid[0] = nb0 * ks0 + nb1 * ks1, out->grid[1] = 1, out->grid[2] = 1;
  out->block[0] = pv->threads(), out->block[1] = 1, out->block[2] = 1;
  out->n_launches = 1;
  out->ks = 1;
  if (int rc = fill_slots(name, out)) return rc;
  set_i32(out, "m", m0), set_i32(out, "k", kk0);
  set_i32(out, "n", n0), set_i32(out, "ks", ks0), set_i32(out, "nb", nb0);
  set_i32(out, "n_b", n1), set_i32(out, "ks_b", ks1), set_i32(out, "nb_b", nb1);
  const saber_iu8_desc *half[2] = {&first, &second};
  for (int h = 0; h < 2; ++h) {
    const char *sfx = h ? "_b" : "";
    const std::string p = std::string("decode_partial") + sfx, c = std::string("decode_counter") + sfx;
    if (half[h]->ks == 1) {
      set_null(out, p.c_str()), set_null(out, c.c_str());
    } else {
      for (uint32_t i = 0; i < half[h]->n_workspaces; ++i) {
        const saber_iu8_workspace &w = half[h]->workspaces[i];
        add_ws(out, (std::string(w.name) + sfx).c_str(), w.kind, strcmp(w.name, "decode_counter") ? w.bytes : (uint64_t)(h ? nb1 : nb0) * 4, w.zero_once);
      }
    }
  }
  return 0;
}

// 33 to 64 rows on the streaming cells' 64-column blocks (iu8_stream_law.h) from three quarters of the CUs, where the 64 x 64
// tile had them. us before / here, W4: 16384 x 5120 at 45 / 64 rows 14.8 / 15.4 -> 11.8 / 13.3, 14336 x 5120 13.8 / 14.7 -> 11.5 / 12.9, x
// 2048 at 40 rows 1.12, x 3072 at 56 rows 1.03 times faster (x 1024 / 2048 0.95 / 1.06); W8 14336 x 4096 at 40 rows 1.08, x 5120 1.06 (x
// 3072 1.02, at 56 rows 0.99).
static bool stream_wide_blocks(bool w8, uint32_t m, uint32_t n, uint32_t k) {
  if (m <= 32 || n <= (CU_COUNT * 3 / 4 - 1) * 64 || n > 64 * CU_COUNT) return false;
  return m <= 48 ? k >= (w8 ? 4096u : 2048u) : !w8 && k >= 3072;
}

// K shares of a streaming launch of 9 to 48 rows. A deep linear of 3,000 to 5,440 columns has too few 64-column blocks for the
// CUs and, on narrower ones, reads its rows once a block: three or four workgroups a block, each on a share of K, divide
// the rows' bytes as well (the partials, shares * M * N * 4 bytes each way, cost some 2 us). us unsplit / here, N = 5120, W4: 16 rows of
// K = 10240 / 12288 / 17408 9.0 / 10.0 / 13.7 -> 8.6 / 9.5 / 11.2 (8192: 7.5 -> 8.0), 32 rows of 8192 / 12288 / 17408 9.1 / 12.5 / 17.4 -> 8.4 /
// 10.3 / 12.7, 48 rows of 8192 / 12288 10.6 / 14.8 -> 9.6 / 11.5 (6144 level); W8 16 / 32 / 48 rows of 12288 14.7 / 17.8 / 20.2 -> 14.2 / 15.2 /
// 16.4. 4096 columns on four shares, 16 / 32 rows of 16384 12.2 / 13.2 -> 11.3 / 11.9, 20 rows of 10240 level. Up to eight rows it is
// level at 5,120 columns and pays on narrower ones of a longer K, which no line takes yet (6 rows, W4 / W8: 3072 x 17408 10.5 / 16.0 -> 8.9 / 12.5,
// 4096 x 17408 10.8 / 16.8 -> 10.1 / 15.0, 3072 x 10240 level / 10.4 -> 9.3). The partials are 3.1 MB at most; a caller without both
// workspaces, saber_iu8_gemm_static and saber_iu8_gemm_pair get the launch in one piece.
static uint32_t stream_split(uint32_t m, uint32_t n, uint32_t k) {
  const uint32_t blocks = (n + 16 * IU8_STREAM_WIDE_NT - 1) / (16 * IU8_STREAM_WIDE_NT);
  const uint32_t z = blocks ? std::min(STREAM_SPLIT_SHARES_MAX, CU_COUNT / blocks) : 0;
  if (m <= STREAM_SPLIT_ROWS_OVER || m > STREAM_SPLIT_ROWS_MAX || z < STREAM_SPLIT_SHARES_MIN || blocks * 4 < CU_COUNT * 3 / 4) return 1;
  return k >= (m <= 16 ? STREAM_SPLIT_K_16ROWS : n <= 4096 ? STREAM_SPLIT_K_4096COLS : STREAM_SPLIT_K) ? z : 1;
}

// The wide streamed cells: blocks of 64, 96 or 144 columns that give three quarters of the CUs and more one block each, from
// the K at which they measured faster than the tile the law had (a short K is all pipeline fill and hand-over in LDS, which
// grow with the block). Before / here in us, K = 5,120 unless it says so -- W4 34816 columns at 24 / 40 / 56 / 72 / 88 rows, ratio 1.18 /
// 1.12 / 1.07 / 1.32 / 1.26; 24576 columns 1.22 / 1.15 / 1.07 / 1.15 / 1.10; 16384 at 72 / 88 rows 1.24 / 1.07; W8 20480 columns 1.37 /
// 1.41 / 1.37 / 1.17 / 1.11, 28672 at 24 / 40 / 56 rows 1.15 / 1.15 / 1.12, 34816 1.07 / 1.03 / 1.03, 14336 at 72 / 88 rows 1.29 / 1.21. One step
// of K below each line: W4 24576 x 1024 at 40 rows 0.93, x 2048 at 56 / 88 rows 0.96 / 0.96; 34816 x 1024 at 40 / 56 / 88 rows 0.96 / 0.86 /
// 0.98; 28672 x 5120 at 40 rows 0.94 (no line there); W8 24576 x 1024 at 72 rows 0.90, 28672 x 2048 at 40 / 56 rows 0.94 / 0.91, 34816 x
// 3072 at 40 rows 1.01. (fifteen widths x six K x five row counts of each kind, weights from memory.)
static const WideVariant *stream_wide_cell(bool w8, uint32_t m, uint32_t n, uint32_t k) {
  if (m <= 16 || m > 96) return nullptr;
  struct Line {
    uint32_t nt, n_over, n_max;  // columns (n_over, n_max]
    uint32_t k4[5], k8[5];       // least K at 17-32, 33-48, 49-64, 65-80, 81-96 rows, int4 / int8 weights; 0: not taken
  };
  constexpr uint32_t BUSY = CU_COUNT * 3 / 4 - 1;
  static const Line LINES[] = {
      {4, BUSY * 64, 64 * CU_COUNT, {0, 0, 0, 8192, 8192}, {0, 0, 0, 2048, 3072}},
      {6, BUSY * 96, 96 * CU_COUNT, {1024, 2048, 4096, 3072, 5120}, {1024, 1024, 2048, 3072, 4096}},
      {9, BUSY * 144, 128 * CU_COUNT, {4096, 0, 0, 0, 0}, {1024, 3072, 4096, 0, 0}},
      {9, 128 * CU_COUNT, 144 * CU_COUNT, {1024, 2048, 4096, 2048, 2048}, {1024, 5120, 8192, 0, 0}},
  };
  const uint32_t tm = (m + 15) / 16;
  for (const Line &l : LINES) {
    if (n <= l.n_over || n > l.n_max) continue;
    const uint32_t k_min = (w8 ? l.k8 : l.k4)[tm - 2];
    return k_min && k >= k_min ? wide_variant(fmt("macaq_iu8_pf_%s_t%ux%u_w", w8 ? "w8" : "w4", tm * 16, l.nt * 16)) : nullptr;
  }
  return nullptr;
}

// The streamed cells on row tiles: outputs of so few 64 x 64 tiles that most CUs idle while a tile goes through its K steps (0.22 us
// each, int4), and streamed launches of so few column blocks that a CU reads every row for one of them. The smallest block that
// is one round of the CUs: 16 x 16, then for int4 16 x 32 and from 65 rows 32 x 32 and 32 x 64. us, the law's pick without these / here, int4,
// K = 5,120: 96 columns at 33 / 64 / 100 / 400 / 777 / 1,500 rows 4.1 / 5.4 / 11.7 / 12.0 / 11.9 / 12.0 -> 3.3 / 4.1 / 5.0 / 5.3 / 6.5 / 8.0, 256 at 200 /
// 777 11.8 / 11.9 -> 5.9 / 8.4, 1024 at 45 / 100 / 200 6.4 / 11.9 / 11.8 -> 5.1 / 7.5 / 8.8, 2048 at 100 11.9 -> 7.9, 5120 at 80 / 96 12.4 / 12.4
// -> 10.2 / 10.4, 512 at 777 12.0 -> 10.4; 96 x 17408 at 400 32.6 -> 11.4, 256 x 1024 at 100 / 777 4.8 / 4.8 -> 3.7 / 3.7.
// Int8: 96 x 5120 at 64 / 200 8.0 / 9.2 -> 5.8 / 6.8, 512 x 5120 at 100 9.3 -> 7.7. Over 240 shapes drawn over the whole of it 16 x 16 1.83 times
// faster, 16 x 32 1.62, 32 x 32 1.45, 32 x 64 1.22, int8 16 x 16 1.32.
// Where the lines lie: up to 48 rows the streamed law has a cell of few columns already: 512 x 2048 at 17 / 45 rows 3.0 / 3.2, here 3.2 /
// 3.5, but 512 x 5120 4.5 / 5.9 -> 4.4 / 5.0 (int8 1024 x 5120 level, 80 x 2432 at 17 rows 3.4 -> 3.5). A second round loses: 16 x 16 on 1024 x 2048
// at 200 rows (832 blocks) 1.02, on 1024 x 5120 at 400 0.64. 32 x 32 on more than 200 blocks at K = 1,024 0.95-1.06; below K = 1,408 it loses where an
// XCD reads many rows and many columns: at 193-256 rows of more than 480 columns 0.86-0.97 up to K = 1,024 and 0.94-1.01 to 1,280 (204 rows of
// 752 x 896 4.5 on 64 x 64, here 5.1), at 161-192 0.93-1.00 and 1.01-1.06, 510 of 368 x 896 0.88, 472 of 352 x 1152 0.91; up to 160 rows 0.98-1.16, up to
// 256 columns 0.98-1.4, from 1,408 on 0.99-1.57; 32 x 64 at K = 2,048 0.93-1.11, at
// 5,120 1.06-1.20, at 17,408 1.23-1.50 (those against 64 x 64 tiles of one wave a wave tile; against their two k-waves 0.94-1.28 at 4,096-6,144, 7 % on average), on more than 208 blocks 0.96 where the 64-row tiles are full (190 rows of 2288 x 5632) and 1.2 where they are
// not (up to 96 rows). Int8 64 x 64 tiles have nothing to unpack: 16 x 32 on 88-160 blocks 0.91-1.32, 7 % on average, not built. Below K = 768 a
// launch is mostly its start (96 x 512 at 100 / 777 rows 3.8 -> 2.8, not taken). Three lines are held: 2,048 rows of 96 x 5120 would gain
// as 1,500 do, 49-64 rows of fewer than 64 columns as 64 columns do, and the tile launches that share K (96 x 17408 at 45 rows 17.0 -> 9.5).
static const RowsVariant *rows_cell(bool w8, uint32_t m, uint32_t n, uint32_t k, bool tile_split) {
  if (m <= ROWS_CELL_ROWS_OVER || m > ROWS_CELL_ROWS_MAX || k < ROWS_CELL_K || k > ROWS_CELL_K_MAX || n > 64 * CU_COUNT || tile_split) return nullptr;
  // an operand past 4 GiB keeps the answer it has without these cells: the streamed form or the tiles' refusal
  if (!tile_operands_hold(w8, m, n, k)) return nullptr;
  auto blocks = [&](uint32_t bm, uint32_t bn) { return (m + bm - 1) / bm * ((n + bn - 1) / bn); };
  // (the variants looked up once)
  static const RowsVariant *const W4_16X16 = rows_variant("macaq_iu8_pf_w4_t16x16_r"), *const W8_16X16 = rows_variant("macaq_iu8_pf_w8_t16x16_r"),
                           *const W4_16X32 = rows_variant("macaq_iu8_pf_w4_t16x32_r"), *const W4_32X32 = rows_variant("macaq_iu8_pf_w4_t32x32_r"),
                           *const W4_32X64 = rows_variant("macaq_iu8_pf_w4_t32x64_r");
  const RowsVariant *const smallest = w8 ? W8_16X16 : W4_16X16;
  if (m <= ROWS_CELL_FEW_ROWS) {
    const bool deep = k >= ROWS_CELL_FEW_DEEP_K;
    const uint32_t widest = w8 ? (deep ? ROWS_CELL_W8_FEW_N : 0) : deep ? ROWS_CELL_FEW_DEEP_N : ROWS_CELL_FEW_N;
    return n <= widest ? smallest : nullptr;
  }
  if (m <= DECODE_MAX_M && n < ROWS_CELL_64_ROWS_N) return nullptr;
  if (blocks(16, 16) <= CU_COUNT) return smallest;
  if (w8) return nullptr;
  if (blocks(16, 32) <= CU_COUNT) return W4_16X32;
  if (m <= DECODE_MAX_M) return nullptr;
  const uint32_t short_rows = k >= ROWS_CELL_32_SHORT_ROWS_K ? ROWS_CELL_32_SHORT_ROWS_DEEP : ROWS_CELL_32_SHORT_ROWS;
  const bool pays_32 = k >= ROWS_CELL_32_SHORT_K || m <= short_rows || n <= ROWS_CELL_32_SHORT_N;
  if (pays_32 && blocks(32, 32) <= (k >= ROWS_CELL_32_K ? CU_COUNT : ROWS_CELL_32_BLOCKS)) return W4_32X32;
  return blocks(32, 64) <= (m <= ROWS_CELL_64_ROWS ? CU_COUNT : ROWS_CELL_64_BLOCKS) && k >= ROWS_CELL_64_K ? W4_32X64 : nullptr;
}

// Which launch `a` and `b` are, whatever their workspaces.
static bool same_launch(const saber_iu8_desc &a, const saber_iu8_desc &b) {
  return !strcmp(a.kernel, b.kernel) && a.ks == b.ks && !memcmp(a.grid, b.grid, sizeof a.grid) && !memcmp(a.block, b.block, sizeof a.block);
}

bool law_split_stream(const saber_iu8_desc &d) {
  int64_t m = 0, n = 0, k = 0;
  const DecVariant *v = dec_variant(d.kernel);
  if (d.ks <= 1 || !v || !int_arg(d, "m", &m) || !int_arg(d, "n", &n) || !int_arg(d, "k", &k)) return false;
  saber_iu8_desc law;
  return !resolve(v->w8 ? SABER_IU8_W8 : SABER_IU8_W4, (uint32_t)m, (uint32_t)n, (uint32_t)k, &law) && same_launch(d, law);
}

// 33 to 64 rows of a deep, narrow int4 linear: the descriptor is the tile launch that shares K (pf_split), and the call that has both
// workspaces in hand streams instead, on as many shares or one fewer: its partials are no more than the tiles', and its arrival
// counters, 16 bits a 64-column block, are a word a 128-column tile. us, tiles / streamed, 33 / 45 / 48 rows of 5120 x 17408 18.2 / 18.8 / 18.4 -> 14.0 /
// 15.3 / 15.1, 50 / 64 19.4 / 19.0 -> 15.9 / 16.4; 40 of 4096 x 17408 18.0 -> 12.8, 64 18.4 -> 14.2; 40 of 3072 x 20480 19.5 -> 12.9. In a pass, behind other kernels, the
// tiles lose 2 us more (four layers of the served graph at 45 rows 372.7 -> 346.2).
bool stream_in_tile_workspaces(const saber_iu8_desc &d, saber_iu8_desc *out) {
  int64_t m = 0, n = 0, k = 0;
  if (strcmp(d.kernel, "macaq_iu8_pf_w4_t64x128_s_ks") || !int_arg(d, "m", &m) || !int_arg(d, "n", &n) || !int_arg(d, "k", &k)) return false;
  if (m > DECODE_MAX_M) return false;
  // (past the rows that the law's own shares end at the lines in columns and K are the same)
  const uint32_t z = stream_split(std::min((uint32_t)m, STREAM_SPLIT_ROWS_MAX), (uint32_t)n, (uint32_t)k);
  if (z <= 1 || z > d.ks) return false;
  // the streamed symbol of the rows and columns (looked up once)
  static const DecVariant *const TM3 = dec_variant("macaq_iu8_dec_w4_tm3"), *const TM3_N2 = dec_variant("macaq_iu8_dec_w4_tm3_n2"),
                          *const TM4 = dec_variant("macaq_iu8_dec_w4_tm4"), *const TM4_N2 = dec_variant("macaq_iu8_dec_w4_tm4_n2");
  const DecVariant *v = n > 16 * CU_COUNT ? (m <= 48 ? TM3_N2 : TM4_N2) : (m <= 48 ? TM3 : TM4);
  if (!iu8_stream_shared_words(false, v->tm, (long)k)) return false;  // (its counters would not fit)
  return !describe_dec(*v, (uint32_t)m, (uint32_t)n, (uint32_t)k, z, out);
}

int unsplit_stream(saber_iu8_desc *d) {
  int64_t m = 0, n = 0, k = 0;
  if (d->ks <= 1 || !dec_variant(d->kernel) || !int_arg(*d, "m", &m) || !int_arg(*d, "n", &n) || !int_arg(*d, "k", &k)) return 0;
  return describe(std::string(d->kernel), (uint32_t)m, (uint32_t)n, (uint32_t)k, 1, d);
}

bool unsplit_pair(const saber_iu8_desc &d, bool bound, bool bound_b, saber_iu8_desc *out) {
  const bool b_first = !strncmp(d.kernel, "macaq_iu8f_pairb_w4_", 20);
  if (!b_first && strncmp(d.kernel, "macaq_iu8f_pair_w4_", 19)) return false;
  static const char *const INTS[] = {"m", "k", "n", "ks", "nb", "n_b", "ks_b", "nb_b"};
  int64_t v[8];
  for (int i = 0; i < 8; ++i)
    if (!int_arg(d, INTS[i], &v[i])) return false;
  const uint32_t m = (uint32_t)v[0], k = (uint32_t)v[1];
  const std::string name = std::string("macaq_iu8_dec_w4_") + (d.kernel + (b_first ? 20 : 19));
  // the halves as the law gives them where they share K, and in one piece where a half shares K without its workspaces
  saber_iu8_desc law[2], now[2], p;
  for (int h = 0; h < 2; ++h) {
    const uint32_t n = (uint32_t)v[h ? 5 : 2], ks = (uint32_t)v[h ? 6 : 3];
    if (ks > 1 ? resolve(SABER_IU8_W4, m, n, k, &law[h]) : describe(name, m, n, k, 1, &law[h])) return false;
    if (law[h].ks != ks) return false;
    now[h] = law[h];
    if (!(h ? bound_b : bound) && unsplit_stream(&now[h])) return false;
  }
  if (pair(law[0], law[1], &p, b_first) || !same_launch(d, p)) return false;
  int64_t w = 0;
  for (int i = 0; i < 8; ++i)
    if (!int_arg(p, INTS[i], &w) || w != v[i]) return false;
  return !pair(now[0], now[1], out, b_first);
}

int resolve(int wkind, uint32_t m, uint32_t n, uint32_t k, saber_iu8_desc *out) {
  if (wkind != SABER_IU8_W4 && wkind != SABER_IU8_W8) return fail(SABER_IU8_E_ARG, "unknown weight kind");
  const bool w8 = wkind == SABER_IU8_W8;
  const char *tag = w8 ? "w8" : "w4";
  if (int rc = check_shape(w8 ? "gemm_i8a8" : "gemm_i4a8", m, n, k)) return rc;
  // The decode band ends where the tile GEMM's small cells overtake the streaming form (speed data of
  // this card: 17..32 rows stream unless the output is very wide, 33..64 unless it is wide; from 49 rows a short K
  // goes to the tiles as well: 8192 x 1024 at 50 / 64 rows 7.4 / 7.6 us streamed, 5.2 / 5.1 on 64 x 64, 5120 x 5120 within
  // a tenth either way, 5120 x 6144 12.2 / 12.5 against 14.1; 4096 x 1024 5.5 against 5.1, 4096 x 4096 8.2 against 10.4).
  // All of it with weights that come from memory, as in a model's pass: at 64 rows streamed / on 64 x 64, int4 4096 x 2048 7.1 / 7.0,
  // 2048 x 3072 7.0 / 8.7, int8 6.3 / 7.2, 7.1 / 9.4; on weights still in the memory-side cache 7.7 / 6.9, 7.6 / 8.7, 6.9 / 5.9,
  // 7.7 / 7.1 (there int8 of up to 3,072 columns would stay on the tiles to K of some 5,000).
  // A deep, narrow linear of int4 weights leaves the band at 33 rows already: where the tile law shares K over workgroups
  // (pf_split), its 64 x 128 cell overtakes the streaming form (5120 x 17408 at 33 / 45 rows on four shares 18.6 / 18.9 us,
  // 21.0 / 22.5 on `tm3_n2`; up to 32 rows streaming wins, 15.5 against 17.5 at 17. A narrower one would stay: 3072 x 16384 at
  // 33 / 45 rows 17.3 / 17.7 shared, 13.7 / 15.0 on `tm3`). The streaming cells' own K shares, which are newer than this line, are faster
  // all over this band at up to 48 rows (stream_split's shares at 40 / 48 rows of 5120 x 17408 14.4 / 15.1, 4096 x 17408 12.8 / 13.3, 3072 x 20480
  // 12.9 / 13.6, on tiles 18.3 / 18.4, 18.0 / 18.0, 19.5 / 19.6): below K = 16,384 they are what the law takes; from there the descriptor
  // stays and saber_iu8_gemm streams in its workspaces (stream_in_tile_workspaces).
  const PfVariant *split_cell = nullptr;
  const uint32_t tile_ks = pf_split(wkind == SABER_IU8_W8, m, n, k, &split_cell);
  if (const RowsVariant *v = rows_cell(w8, m, n, k, tile_ks && m > 32)) return describe_rows_cell(*v, m, n, k, out);
  const bool narrow = n <= 16 * CU_COUNT, two_wide = !narrow && n <= 32 * CU_COUNT;  // a 16- / 32-column block a CU
  const bool stream = m <= 16 || (m <= 32 && n <= 16384) || (m <= 48 && n <= 8192 && tile_ks == 0) ||
                      (tile_ks == 0 && m <= 64 && stream_wide_blocks(w8, m, n, k)) ||
                      (tile_ks == 0 && ((narrow && k >= 2048) || (two_wide && k >= 6144)));
  if (m <= DECODE_MAX_M && stream) {
    // Up to 16 rows of K <= 5120: the persistent form that stages the 16-row tile once a workgroup (`_s80`) where
    // it measured faster than the streamed one, which re-reads the tile from L2 once a 32-column block. W4, 9-16
    // rows: everywhere (gate+up 34816 x 5120 19.1 -> 16.6 us, 28672 x 4096 13.2 -> 12.1, 14336 x 5120 9.4 -> 9.0,
    // QKV / O 6.1 / 5.9 -> 6.05 / 5.8); up to 8 rows, and int8 weights at any row count, from 64 MiB of weights
    // (W4 5-8 rows: gate+up 16.6-17.9 -> 16.4-17.2, 28672 x 4096 even, 14336 x 5120 8.5 -> 9.0 the other way;
    // W8: gate+up 31.3 -> 28.4, 28672 x 4096 21.0 -> 19.9, 14336 x 5120 14.3 -> 13.6, QKV 8.1 -> 8.4 the other way).
    // A wide N (from 24,576 columns: three and more column blocks a workgroup) takes it at any row count, also against the
    // staged 20 KiB form of 1-4 rows, which starts a workgroup a block (W4 gate+up at 1 / 2 / 4 rows 17.6 / 16.4 / 16.7 ->
    // 16.6 / 15.8 / 16.35, 24576 x 2048 7.5-7.6 -> 6.85-6.9, 28672 x 4096 12.1-12.25 -> 11.2-11.9; W8 gate+up 29.2-30.8 ->
    // 27.9-29.0; at 14336 columns and fewer it loses 0.1-0.7 us there).
    if (k <= 5120 && staged80_holds(m, k) &&
        ((m > 8 && wkind == SABER_IU8_W4) || n >= S80_MIN_N ||
         (m > 4 && (uint64_t)n * k / (wkind == SABER_IU8_W8 ? 1 : 2) >= S80_MIN_BYTES)))
      return describe_s80(wkind == SABER_IU8_W8, false, m, n, k, 1, out);
    // ... and 2 to 4 rows of a long K, whose live rows' codes fit the same 80 KiB (the copy takes their pieces of the
    // tile): 5120 x 17408 at 2 / 3 / 4 rows 11.0 -> 10.5 / 10.7 / 10.7 us; at K = 6144 and 8704 (5.7 -> 5.8, 6.9 -> 6.9)
    // and on 16384 x 8192 (12.4 -> 12.8) the streamed form stays
    if (m >= 2 && m <= 4 && k >= 16384 && wkind == SABER_IU8_W4 && staged80_holds(m, k))
      return describe_s80(false, true, m, n, k, 1, out);
    // 17 to 64 rows: the block width that gives every CU one column block (iu8_variants.def has the timings). 33 to 48
    // rows keep `tm3` at a short K (8192 x 1024 at 40 rows 6.1 us against 6.2 on `_n2`).
    std::string name = dec_stream_name(tag, m, k);
    if (m > 16 && m <= 32 && narrow) name += "_n1";
    else if (m > 32 && two_wide && k >= 4096) name += "_n2";
    else if (m > 48 && narrow) name += "_k16";
    const DecVariant *v = dec_variant(name);
    if (!v) return fail(SABER_IU8_E_RULE, name + ": no such variant");
    return describe_dec(*v, m, n, k, stream_split(m, n, k), out);
  }
  if (const WideVariant *v = stream_wide_cell(w8, m, n, k)) return describe_wide(*v, m, n, k, out);
  if (tile_ks) return describe_pf(*split_cell, m, n, k, tile_ks, out);
  // One row tile, past the streaming band: a tile's chain of K steps is what the launch takes, so the cell is the
  // narrowest that needs one round of the 256 CUs (the estimate of pf_cell is fitted to 65 rows and more and took 64 x 64
  // up to 32,768 columns: two rounds). W4, us on 64 x 64 / 64 x 128 at 17 / 45 / 64 rows: 20480 x 5120 18.6 / 20.6 / 22.5 ->
  // 15.0 / 16.3 / 17.2, 28672 x 5120 20.3 / 22.4 / 24.4 -> 16.8 / 18.0-20.6 / 18.6-19.3, 24576 x 2048 at 20 / 50 rows
  // 10.3 / 11.4 -> 8.8 / 9.2; at 32768 columns 23.4 / 23.6 / 25.3 -> 19.6 / 23.7 / 24.8; up to 16,384 columns 64 x 64 is one
  // round (16384 x 5120 13.5 against 15.6-16.7) and pf_cell's pick. 160 columns wide up to 40,960 columns (40960 x 5120 at 17 /
  // 33 / 64 rows 29.6 / 32.5 / 33.5 -> 24.8 / 28.9 / 30.2, W8 52.9 / - / 57.0 -> 42.0 / - / 41.6). There is no line in K: a K of
  // 512 and less, which no decoder linear this wide has, is 3-23 % slower on the 160-column cells (32784 x 256 at 33 rows W4
  // / W8 +17 / +12 %; W4 level from 1,024 there and from 640 at 34,816 columns and more, W8 from 384; 36864 columns W4 +8 %, W8
  // faster). Int8 weights up to 32,768 columns stay with the estimate
  // (64 x 64 and 64 x 128 within 10 % of each other).
  if (m <= 64 && n > 32 * 2 * CU_COUNT && n <= 160 * CU_COUNT) {
    const char *cell = n > 128 * CU_COUNT ? (!w8 && m <= 32 ? "t32x160_s" : "t64x160_s") : w8 ? nullptr : "t64x128_s";
    if (cell) return describe_pf(*pf_variant(fmt("macaq_iu8_pf_%s_%s", tag, cell)), m, n, k, 0, out);
  }
  // Int8 weights: 128 x 160 where it is one round and 128 x 128 is two; us against the estimate's pick -- 5120 x 17408 at
  // 777 / 1,000 rows 121 / 122 -> 91 / 96, 5120 x 5120 42.4 / 40.6 -> 30.6 / 33.0, 10240 x 5120 at 400 / 512 rows 41 / 42 ->
  // 33 / 35, 6144 x 5120 at 700 rows 39.5 -> 35.7, 20480 x 5120 at 130 / 200 rows 37.7 / 45.1 -> 36.1 / 37.5. One round of
  // both (5120 columns at 700 rows, 25.8 against 32.6) and two of both (8192 x 8192 at 777, 67 against 90) are the
  // estimate's. Where the estimate has a 64-row cell (the rows' last block of 128 is at most half live), from K = 5,120:
  // 18432 x 1024 / 2048 / 4096 / 5120 at 129 rows 12.0 / 18.7 / 28.8 / 36.3 there, 11.6 / 17.0 / 27.7 / 32.6 here, but
  // 7168 x 1024 / 2048 / 4096 / 5120 at 513 rows 12.0 / 16.7 / 29.1 / 37.8 against 13.6 / 20.1 / 30.1 / 39.6 and every
  // such launch of K <= 256 4-24 % slower here; of 466 timed at K = 5,120 and 6,144 eight are 3-5 % slower, the rest up to 40 %
  // faster. Where it has a larger cell: a tile count that is not whole eighths leaves the order by XCD (iu8_dense_tile_at),
  // which costs what the round saves at K of 512 to 2,048 (1024 deep, 5760 columns at 784 rows 13.3 -> 15.2, 5632 columns,
  // 216 tiles, at 720 rows 13.5 -> 11.0); one row block never lost. 1,024 rows and more stay with the
  // estimate, whose table does not hold this cell: not for its speed at 1,024 rows themselves, where it is as many tiles as
  // at 1,000 (5120 x 5120 / 17408 32.6 / 99 us, 128 x 256 41.2 / 118); from 1,025 rows of 5,120 columns it is two rounds
  // (55.4 / 174 against 42.4 / 124).
  // Int8 weights where the estimate, whose rates rank a 64-row cell too high past one round of it, has such a cell: 128 x 64 where that is one
  // round and 64 x 64 is not (a 64 x 128 tile, the estimate's pick of a long K, has as many bytes and half the rows to share a weight stage), else
  // 128 x 128 where that is one and 64 x 128 is not. us, the estimate's pick / here: 200 rows of 5120 x 17408 / 6144 / 5120 62.8 / 23.4 / 21.2 -> 47.0 /
  // 18.7 / 17.0, 300 of 4096 x 17408 61.5 -> 46.3, 160 of 7168 x 5120 22.0 -> 17.3, 777 of 2048 x 17408 59.8 -> 48.0, 300 of 5120 x 3072 14.7 -> 11.6; 160 / 256 of
  // 16384 x 5120 36.9 / 39.4 -> 29.3 / 32.4, 227 of 16384 x 4096 1.25, 152 of 14336 x 256 1.26 times faster. From K = 2,048 (2,048 level to 1.11, 3,072 1.07-1.27, 5,120
  // and more 1.05-1.38, 1,024 0.95-1.05), from 4,096 on a count that is not whole eighths (854 rows of 1776 x 3072 0.88); with no more 64 x 64 tiles than
  // CUs those stay (160 of 5120 x 3072 0.80). Over 305 shapes of 65 to 4,096 rows that moved, drawn after the lines, 128 x 64 1.20 times faster, 128 x 128 1.26, the
  // slowest 0.99. 256 rows are held on the 64 x 128 cell (5120 x 5120 / 6144 / 17408 21.7 / 24.7 / 63.5 for 18.9 / 21.5 / 53.1).
  if (w8 && m > 64) {
    auto tiles = [&](uint32_t bm, uint32_t bn) { return (uint64_t)((n + bn - 1) / bn) * ((m + bm - 1) / bm); };
    static const PfVariant *const T128X160 = pf_variant("macaq_iu8_pf_w8_t128x160"), *const T128X64 = pf_variant("macaq_iu8_pf_w8_t128x64_s"),
                           *const T128X128 = pf_variant("macaq_iu8_pf_w8_t128x128");
    const PfVariant *est = pf_cell(w8, m, n, k);
    const bool small = est->block_m() == 64;
    const bool pays = small ? k >= 5120 : m <= 128 || k < 512 || k >= 3072 || tiles(128, 160) % 8 == 0;
    if (m < 1024 && pays && tiles(128, 160) <= CU_COUNT && tiles(128, 128) > CU_COUNT) est = T128X160;
    else if (small && tiles(128, 64) <= CU_COUNT) {
      if (m != 256 && tiles(64, 64) > CU_COUNT && k >= (tiles(128, 64) % 8 ? 4096u : 2048u)) est = T128X64;
    } else if (small && tiles(128, 128) <= CU_COUNT && tiles(64, 128) > CU_COUNT) {
      est = T128X128;
    }
    return describe_pf(*est, m, n, k, 0, out);
  }
  return describe_pf(*pf_cell(wkind == SABER_IU8_W8, m, n, k), m, n, k, 0, out);
}

// K shares of a tile launch (0: none). A deep, narrow linear at a few dozen rows gives the unsplit
// law so few tiles that half to two thirds of the CUs idle through hundreds of K steps; there, 2-4 workgroups
// a tile of the 64x128 cell, each on a share of K, are faster although the partials travel through memory (ks * M * N * 4
// bytes each way, and the last share to arrive sums the others). The launch then needs the `decode_partial` /
// `decode_counter` workspaces the descriptor lists.
uint32_t pf_split(bool w8, uint32_t m, uint32_t n, uint32_t k, const PfVariant **cell) {
  // us, the law's shares against the fastest unsplit cell: 5120 x 17408 at 64 / 128 / 160 / 192 rows 19.4 / 22.4 / 28.8 / 29.3
  // against 24.6 / 33.5 / 33.5 / 33.8, at 200 / 256 rows three shares 37.4 / 38.1 against 35.4 / 39.6; 8192 x 16384 at 96 / 128 rows
  // 27.7 / 28.7 against 32.4 / 33.1, and past 128 tiles, at 160 rows, 49.9 against 35.2; 3072 x 16384 at 160 / 192 rows 21.1 / 21.1
  // against 31. The lines in K and rows were drawn with a slower reduction and are narrower than these timings would have
  // them: K = 12,288 is not shared (5120 columns at 96 / 128 / 192 rows 18.0 / 18.3 / 22.1 on shares, 24.6 / 24.8 / 25.2 as it
  // is), nor 96 tiles at 200-256 rows (3072 x 16384 25.7 against 31.5), nor 2-4 tiles of K = 5,120 (96 columns at 96-256
  // rows 10.0 against 11.6); six shares of 40 tiles are 2-3 % ahead of four at 33-64 rows, eight behind. (A `_ks`
  // workgroup takes 81,924 bytes of LDS: one a CU, not the two of `occ`.)
  if (w8 || k < 16384 || m > 192) return 0;
  const PfVariant *v = pf_variant("macaq_iu8_pf_w4_t64x128_s");
  if (!v || !signature_for(std::string(v->name) + "_ks")) return 0;
  const uint64_t tiles = (uint64_t)((n + v->block_n() - 1) / v->block_n()) * ((m + v->block_m() - 1) / v->block_m());
  if (tiles > 128) return 0;
  *cell = v;
  return (uint32_t)std::min<uint64_t>(4, CU_COUNT / tiles);
}

// The prefill cell of a shape: the tile whose estimated time is least. A launch's time is a fixed
// cost, a cost a tile the busiest workgroup runs (pipeline fill, epilogue, tile switch: what a cell pays
// whatever K is) and the largest of three: the matrix work of the busiest CU over the cell's measured rate
// (co-resident workgroups of a two-a-CU cell share the CU's matrix units), the bytes that CU pulls in
// (its tiles' A rows and W columns, K deep) over what one CU takes from L2, and all tiles' bytes over
// what the L2s deliver together -- the last two are what bind for M up to about 512, where the A rows
// are re-read once a column block, so small tiles that put every CU to work win there and the large
// ones take over as the matrix work grows -- or the weights' way from memory, once for every row tile
// that runs beside another on the same column block (the wide gate+up at 256 rows on 128-row tiles). The constants are this card's speed data, one table a weight
// kind (int8 weights are twice the bytes a tile and have no unpack: the cells rank differently), fitted to
// sustained timings of every cell on the four 27B-class shapes x 14 row counts from 65 to 8,192, weights
// cold (successive launches walk copies that exceed the memory-side cache; with warm weights the 64 x 64
// cell overtakes the 64 x 128 one at 256 rows, which no layer of a model sees), and checked on shapes the fit had
// not seen -- the served 27B graph's own 16384 x 5120, 14336 x 5120, 5120 x 6144 and 96 x 5120 at eight row counts,
// which moved three small-cell rates and took the side-by-side term off the 64-row cells.
// The W4 rates are a fit to 2,549 shapes of 65 to 8,192 rows, 256 to 35,200 columns and K of 128 to 17,408, spread over the logarithm of
// each and over the served widths, every cell timed on weights from memory; what it minimises is the time of the cell it picks
// over the fastest one's, with three times the weight on what a shape loses against its pick before. The pick takes 0.9 % more than
// the fastest cell over them (3.4 % with the rates before, which were drawn when the 128- and 256-row cells got their k-waves from
// shapes with few short K among them, and took slower cells than the ones in use there: 611 rows of 14368 x 768 20.2 us on 128 x
// 320 for 16.0 on 256 x 256, 125 of 288 x 128 3.6 on 64 x 128 for 3.2 on 64 x 64, 217 of 25984 x 2304 26.5 on 128 x 128 for 24.0). On 814
// other shapes where the pick has moved it is 5 % faster than those rates' and 6 % than the ones' before the k-waves; slower than
// either by more than 4 % on nine, three of them past a K of 17,408 (3,324 rows of 2016 x 18688 123 -> 140) and two of about 1,350 rows
// of 14336 x 1024 (31 -> 33). 634 rows of 12160 x 2688 take 28.3 on 128 x 128 two a CU (28.5 on 128 x 256 as it was, 24.6 as it is).
// 128 x 256 is held up to 1,023 rows (600 rows of 34816 x 5120 113 there, 119 on the pick, 126 before; 777 of 5120 x 17408 92 for 96):
// from 1,024 the pick of a narrow output is 128 x 128 two a CU as before, although 128 x 256 has become 5 % faster (1,024 / 1,100 /
// 1,300 rows of 5120 x 17408 100 / 103 / 119 against 95 / 98 / 110): there one rate cannot keep both. W8, output-side shapes
// from 2,048 rows: every pick the fastest; at 1,025 to 1,280 rows up to 7 % off (256 x 160, 128 x 128 two a CU). The
// reference keeps its band tables the same way
// (crates/saber-kernels/src/macaq_iu8.rs:150-212). One table for both kinds had sent the int8-weight
// O and down projections at 2,048 rows to the 128 x 320 cell, 17-22 % behind the 256 x 160 cell there.
const PfVariant *pf_cell(bool w8, uint32_t m, uint32_t n, uint32_t k) {
  // rows: the cell is held for launches of fewer (0: of any count)
  struct Cell { const char *tile; double tops_per_cu, tile_us; uint32_t rows; };
  // quarter: the rate of the 128 x 128 tiles in the 256 x 256 cell's last round (held while the others were fitted)
  struct Law { double fixed_us, cu_gbps, l2_tbps, lone, hbm_tbps, side_cap, quarter; Cell cells[10]; };
  static const Law W4 = {1.729, 90.000, 14.830, 23.134, 4.944, 2.018, 8.799,
                         {{"tn4_lbk64", 13.270, 1.444}, {"t256x320", 12.890, 2.969}, {"t128x320", 12.932, 5.553}, {"t256x160", 11.387, 3.577}, {"t128x128", 7.955, 0.429}, {"t128x128_o2", 9.929, 0.709}, {"t64x128_s", 7.719, 0.442}, {"t64x64_s", 4.276, 0.226}, {"t128x256", 13.391, 9.456, 1024}}};
  // up to 64 rows, which the lines above this estimate in `resolve` are drawn against
  static const Law W4_64 = {0.974, 90.000, 19.875, 1.422, 3.113, 2.116, 8.799,
                            {{"tn4_lbk64", 14.007, 3.223}, {"t256x320", 13.568, 4.138}, {"t128x320", 11.147, 7.968}, {"t256x160", 11.173, 8.857}, {"t128x256", 9.046, 1.844}, {"t128x128", 8.799, 2.045}, {"t128x128_o2", 9.622, 3.231}, {"t128x64_s", 4.711, 1.952}, {"t64x128_s", 6.085, 2.027}, {"t64x64_s", 5.582, 1.829}}};
  static const Law W8 = {4.419, 75.175, 18.116, 1.782, 5.234, 1.935, 8.069,
                         {{"tn4_lbk64", 13.145, 0.244}, {"t256x320", 12.800, 0.000}, {"t128x320", 6.328, 2.194}, {"t256x160", 11.499, 0.000}, {"t128x256", 10.761, 3.251}, {"t128x128", 8.069, 0.427}, {"t128x128_o2", 8.619, 0.229}, {"t128x64_s", 4.123, 0.073}, {"t64x128_s", 6.003, 2.817}, {"t64x64_s", 5.960, 0.000}}};
  const Law &law = w8 ? W8 : m <= 64 ? W4_64 : W4;
  // the cells' variants, looked up once
  constexpr size_t NCELL = sizeof(Law::cells) / sizeof(Cell);
  using Variants = std::array<const PfVariant *, NCELL>;
  auto variants = [](const Law &l, const char *tag) {
    Variants v{};
    for (size_t i = 0; i < NCELL && l.cells[i].tile; ++i) v[i] = pf_variant(fmt("macaq_iu8_pf_%s_%s", tag, l.cells[i].tile));
    return v;
  };
  static const Variants V4 = variants(W4, "w4"), V4_64 = variants(W4_64, "w4"), V8 = variants(W8, "w8");
  const Variants &cells = w8 ? V8 : m <= 64 ? V4_64 : V4;
  const PfVariant *best = nullptr;
  double best_t = 0;
  for (size_t i = 0; i < NCELL; ++i) {
    const Cell &c = law.cells[i];
    const PfVariant *v = cells[i];
    if (!v || (c.rows && m >= c.rows)) continue;
    const double bm = v->block_m(), bn = v->block_n();
    const uint64_t tiles = (uint64_t)((n + v->block_n() - 1) / v->block_n()) * ((m + v->block_m() - 1) / v->block_m());
    const uint64_t grid = std::min<uint64_t>(tiles, (uint64_t)CU_COUNT * v->occ);
    const uint64_t per_wg = (tiles + grid - 1) / grid;
    double cu_tiles = (double)per_wg * std::min<uint64_t>(v->occ, (grid + CU_COUNT - 1) / CU_COUNT);
    // the 256 x 256 cell runs a thin last round (at most half the workgroups) as quarter tiles on the
    // 128 x 128 cell, each a quarter of the work at that cell's rate
    const uint64_t q = tiles / grid, rem = tiles - q * grid;
    if (!strcmp(c.tile, "tn4_lbk64") && q >= 1 && rem > 0 && 2 * rem <= grid)
      cu_tiles = (double)q + (double)((4 * rem + grid - 1) / grid) * 0.25 * (c.tops_per_cu / law.quarter);
    // ... and a few rows past the last whole 256 as thin tiles (int4 weights: the estimate of the int8 cells is drawn without)
    if (!strcmp(c.tile, "tn4_lbk64") && !w8 && tiles < (1u << 20) && k < (1u << 30)) {
      const iu8_pf_plan plan = iu8_pf_plan256((int)m, (int)((n + 255) / 256), (int)grid, (int)k, w8);
      if (plan.thin) cu_tiles = std::min(cu_tiles, plan.cost * 0.0101);  // (in tiles, with the fit's factor)
    }
    const double tile_bytes = bm * k + bn * k * (w8 ? 1.0 : 0.5);
    const double t_mfma = cu_tiles * bm * bn * k * 2.0 / (c.tops_per_cu * 1e6);
    const double t_cu = cu_tiles * tile_bytes / (law.cu_gbps * 1e3);
    const double t_l2 = (double)tiles * tile_bytes / (law.l2_tbps * 1e6);
    // the two-a-CU 128 x 128 cell alone on a CU (no more workgroups than CUs) has four waves to hide
    // its latencies with and measured well behind the eight-wave 128 x 128 cell there
    const double lone = !strcmp(c.tile, "t128x128_o2") && grid <= CU_COUNT ? law.lone : 1.0;
    // cold weights: the row tiles that run side by side on one column block each fetch it from memory -- those of the
    // 128- and 256-row cells; the 64-row cells' neighbours share a column block's lines (fetch over operands 1.5-1.65 at
    // four row tiles by the counters, and the wide projections of the served graph at 65-128 rows: 16.5-18.8 us on
    // 64 x 128 where a doubled fetch would make it 27)
    const uint64_t gx = (n + v->block_n() - 1) / v->block_n(), gy = (m + v->block_m() - 1) / v->block_m();
    const double side = v->block_m() == 64 ? 1.0 : std::min<double>((double)std::min<uint64_t>(gy, std::max<uint64_t>(1, grid / gx)), law.side_cap);
    const double t_hbm = ((double)n * k * (w8 ? 1.0 : 0.5) * side + (double)m * k) / (law.hbm_tbps * 1e6);
    const double t = law.fixed_us + (double)per_wg * c.tile_us + lone * std::max(std::max(t_mfma, t_hbm), std::max(t_cu, t_l2));
    if (!best || t < best_t) best = v, best_t = t;
  }
  return best;
}

static int describe_rows(const char *op, const char *kernel, uint32_t rows, uint32_t width, const char *wname,
                         saber_iu8_desc *d) {
  if (rows == 0 || width == 0) return fail(SABER_IU8_E_RULE, fmt("%s: %u rows of %u has nothing to do", op, rows, width));
  if (width % 64 != 0 || width > 32768)
    return fail(SABER_IU8_E_RULE, fmt("%s: row width %u must be a multiple of 64 (whole A fragments), at most 32768", op, width));
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_i8q");
  copy_name(d->kernel, sizeof d->kernel, kernel);
  // the wave-a-row forms take four rows a workgroup
  const bool w64 = strlen(kernel) > 4 && !strcmp(kernel + strlen(kernel) - 4, "_w64");
  if (w64 && (rows % 4 != 0 || width > 4096))
    return fail(SABER_IU8_E_RULE, fmt("%s: %s takes a multiple of 4 rows of at most 4096, got %u of %u", op, kernel, rows, width));
  const bool t1024 = strlen(kernel) > 6 && !strcmp(kernel + strlen(kernel) - 6, "_t1024");
  d->grid[0] = w64 ? rows / 4 : rows, d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = t1024 ? 1024 : 256, d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(kernel, d)) return rc;
  set_i32(d, wname, width);
  return 0;
}

// The fused forms quantise rows whose int8 codes (rows rounded up to a power of two) fit the kernel's
// staging area: up to 4 rows in 20 KiB (`_tm1`), up to 16 rows in 80 KiB (`_tm1_a80`). Every workgroup
// repeats the rows' quantisation (about 0.5 us a row of 5,120 on this card), a producer launch costs
// about 3 us once. The kernel itself holds what `fused_form_holds` says, by name; what the law launches is
// `fused_holds` below.
static uint64_t staged_bytes(uint32_t m, uint32_t k) {
  uint32_t mr = 1;
  while (mr < m) mr *= 2;
  return (uint64_t)mr * k;
}
bool fused_small_holds(uint32_t m, uint32_t k) { return m >= 1 && m <= 4 && staged_bytes(m, k) <= 20 * 1024; }
bool fused_form_holds(bool a80, uint32_t m, uint32_t k) {
  return a80 ? m >= 1 && m <= 16 && staged_bytes(m, k) <= 80 * 1024 : fused_small_holds(m, k);
}
// the MLP chain: the first linear's rows (hidden wide) in the 20 KiB form, the second's (intermediate wide) in
// the 20 KiB form or, for up to 4 rows, the 80 KiB one
bool mlp_chain_form_holds(uint32_t m, uint32_t hidden, uint32_t inter) {
  return fused_small_holds(m, hidden) && (fused_small_holds(m, inter) || (m <= 4 && fused_form_holds(true, m, inter)));
}
// Where the one launch beats the three (fused gate+up linear, 16-wave activation producer, streamed down GEMV), graph
// replay on cold weights, hidden / intermediate in us chain / three: one row 5120/17408 32.9/34.2, 5120/13824 27.4/29.2,
// 4096/14336 25.5/27.0, 4096/12288 23.0/24.2, 8192/8192 25.9/25.8, 5120/5120 18.9/17.5; two rows 5120/17408 35.3/36.0,
// 5120/13824 29.9/30.9, 4096/14336 28.0/28.7, 4096/12288 25.7/25.4; three rows 36.5-36.8/36.6-37.4 and 31.9/31.6; four
// rows 38.2/37.3, 33.7/32.6, 28.6/26.2. (A meeting inside the launch costs more than the gap between two launches;
// what the chain saves is the activation's pass over memory and one launch.)
bool mlp_chain_pays(uint32_t m, uint32_t hidden, uint32_t inter) {
  if (inter > 20 * 1024) return false;  // not measured past the one-row form's 20 KiB of codes
  return mlp_chain_form_holds(m, hidden, inter) && ((m == 1 && inter >= MLP_CHAIN_PAYS_INTER_1) || (m == 2 && inter >= MLP_CHAIN_PAYS_INTER_2));
}
// The law: the 20 KiB form wherever it holds (1-4 rows: 5.7 / 5.3 / 16.7 us against 7.8 / 7.2 / 19.7 as two launches
// at one row of the 27B layer's K = 5120 shapes, 6.9 / 6.7 / 17.2 against 8.0 / 7.5 / 19.2 at four); the 80 KiB form at
// two rows of K >= 16384 (K = 17408: 13.85 against 13.98 us, and a launch fewer); elsewhere it loses to the 16-wave
// producer + the streamed or staged GEMV (two rows of K = 12288: 11.4 / 11.2; three rows of K = 17408: 14.8 / 14.1, of
// 8192: 10.0 / 9.5; four rows: 16.0 / 14.8 at K = 17408, 10.5 / 9.5 at 8192, 9.2 / 8.5 at 6144).
bool fused_holds(uint32_t m, uint32_t k) {
  return fused_small_holds(m, k) || (m == 2 && k >= FUSED_A80_MIN_K && fused_form_holds(true, m, k));
}

uint32_t fused_grid(uint32_t nblk) {
  if (nblk <= CU_COUNT) return nblk;
  const uint32_t per = std::min<uint32_t>(8, (nblk + CU_COUNT - 1) / CU_COUNT);
  return (nblk + per - 1) / per;
}

int resolve_fused(int wkind, uint32_t m, uint32_t n, uint32_t k, saber_iu8_desc *d) {
  if (wkind != SABER_IU8_W4 && wkind != SABER_IU8_W8) return fail(SABER_IU8_E_ARG, "unknown weight kind");
  const char *op = wkind == SABER_IU8_W8 ? "linear_i8a8_fused" : "linear_i4a8_fused";
  if (int rc = check_shape(op, m, n, k)) return rc;
  if (!fused_holds(m, k))
    return fail(SABER_IU8_E_RULE, fmt("%s: %u rows of %u are not a fused launch (up to 4 rows in 20 KiB of codes; 2 rows of K >= 16384 in 80 KiB)", op, m, k));
  // one long row: the form that makes the row's codes just in time inside the weight stream (`_r1`). Measured on
  // this card against the several-row form at one row (cold weights, graph replay, N = 5120): K = 8,192 6.47
  // against 6.91 us, 12,288 7.82 against 8.38, 17,408 9.88 against 10.7-11.4, 20,480 10.97 against 11.83; at
  // K = 5,120 it loses (5.64 against 5.17: there a thread of the several-row form converts one piece at most,
  // which is what this form's first chunk costs, and its two column groups convert every piece twice)
  const std::string name = m == 1 && k >= FUSED_R1_MIN_K && fused_small_holds(m, k)
                               ? fmt("macaq_iu8_decq_%s_r1", wkind == SABER_IU8_W8 ? "w8" : "w4")
                               : fmt("macaq_iu8_decq_%s_tm1%s", wkind == SABER_IU8_W8 ? "w8" : "w4", fused_small_holds(m, k) ? "" : "_a80");
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8");
  copy_name(d->kernel, sizeof d->kernel, name);
  // 16 waves: 8 k-waves x 2 weight tiles = 32 columns a block, one workgroup a CU. Past one block a
  // CU the workgroups walk the blocks in equal shares (1,088 blocks: 218 workgroups x 5, measured 15.8 us
  // against 16.2 on 256 workgroups with 4 or 5), at most 8 each (the kernel's scale table).
  d->grid[0] = fused_grid((n + 31) / 32), d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = 1024, d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", n);
  set_i32(d, "k", k);
  return 0;
}

// The decode MLP as one persistent launch (kernels/iu8_chain.h): both linears in the fused form's
// bounds, every workgroup resident at once (two a CU: the runtime checks what the card really
// holds), at most 8 column blocks of either linear a workgroup.
int resolve_mlp_chain(uint32_t m, uint32_t hidden, uint32_t inter, uint32_t spin, saber_iu8_desc *d) {
  const char *op = "mlp_chain_i4a8";
  if (inter > 0x3FFFFFFFu) return fail(SABER_IU8_E_RULE, fmt("%s: intermediate width %u", op, inter));
  if (int rc = check_shape(op, m, 2 * inter, hidden)) return rc;
  if (int rc = check_shape(op, m, hidden, inter)) return rc;
  if (!mlp_chain_form_holds(m, hidden, inter))
    return fail(SABER_IU8_E_RULE, fmt("%s: %u rows of %u / %u do not fit the fused form (at most 4 rows, 20 KiB of codes at the hidden "
                                      "width, 80 KiB at the intermediate)", op, m, hidden, inter));
  // the first linear walks inter / 16 paired tiles, the second hidden / 32 column blocks; one workgroup a CU
  const uint32_t nblk = std::max(inter / 16, (hidden + 31) / 32);
  if (nblk > 8 * CU_COUNT)
    return fail(SABER_IU8_E_RULE, fmt("%s: %u column blocks are more than the %u resident workgroups walk (8 each)", op, nblk, CU_COUNT));
  const uint32_t grid = std::max(fused_grid(inter / 16), fused_grid((hidden + 31) / 32));
  // the second linear's rows in 20 KiB of staged codes, else in 80 KiB (`_a80`: 2 to 4 rows of the 27B layer's 17,408)
  const char *name = fused_small_holds(m, inter) ? "macaq_iu8f_mlp_w4_tm1" : "macaq_iu8f_mlp_w4_tm1_a80";
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8f");
  copy_name(d->kernel, sizeof d->kernel, name);
  d->grid[0] = grid, d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = 1024, d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "k", hidden);
  set_i32(d, "n", inter);
  set_i32(d, "spin", spin ? spin : MLP_CHAIN_SPIN);
  add_ws(d, "p", SABER_IU8_WS_SCRATCH, (uint64_t)m * inter * 2, 0);
  add_ws(d, "state", SABER_IU8_WS_PERSISTENT, MLP_CHAIN_STATE_BYTES, 1);
  return 0;
}

// The gate+up linear of a decode MLP with SiLU(gate) * up in its epilogue (`macaq_iu8f_gateup_act_w4_s80`): the rows'
// 16-row tile staged once a workgroup (what `_s80` holds), a column block = one 16-column tile of p.
bool gate_up_act_holds(uint32_t m, uint32_t hidden, uint32_t inter) {
  return m >= 1 && m <= 16 && hidden % 128 == 0 && inter % 16 == 0 && inter > 0 && staged80_holds(m, hidden) && inter / 16 <= 8 * CU_COUNT;
}
int resolve_gate_up_act(uint32_t m, uint32_t hidden, uint32_t inter, saber_iu8_desc *d) {
  const char *op = "linear_i4a8_gate_up_act";
  if (inter > 0x3FFFFFFFu) return fail(SABER_IU8_E_RULE, fmt("%s: intermediate width %u", op, inter));
  if (int rc = check_shape(op, m, 2 * inter, hidden)) return rc;
  if (!gate_up_act_holds(m, hidden, inter))
    return fail(SABER_IU8_E_RULE, fmt("%s: %u rows of %u / %u: at most 16 rows whose codes (rows rounded up to a power of two) fit 80 KiB, "
                                      "at most %u tiles of 16 columns", op, m, hidden, inter, 8 * CU_COUNT));
  const char *name = "macaq_iu8f_gateup_act_w4_s80";
  memset(d, 0, sizeof *d);
  copy_name(d->op, sizeof d->op, op);
  copy_name(d->plugin, sizeof d->plugin, "macaq_iu8f");
  copy_name(d->kernel, sizeof d->kernel, name);
  d->grid[0] = fused_grid(inter / 16), d->grid[1] = 1, d->grid[2] = 1;
  d->block[0] = 1024, d->block[1] = 1, d->block[2] = 1;
  d->n_launches = 1;
  d->ks = 1;
  if (int rc = fill_slots(name, d)) return rc;
  set_i32(d, "m", m);
  set_i32(d, "n", inter);
  set_i32(d, "k", hidden);
  return 0;
}

// The row kernels' register forms: the narrowest that holds the row (4,096 elements a group slot).
// Many narrow rows go a wave a row (`base`_w64), the rest a workgroup a row (`base`_t256...).
// Rows wider than 4,096 whose count leaves the card part idle go 16 waves a row (`base`_t1024): measured on this
// card, graph replay, 256-thread form / 1024-thread form in us -- the quantiser at 1 / 16 / 256 rows of 5,120:
// 2.57/2.34, 2.98/2.74, 3.41/3.20; of 17,408: 3.90/2.91, 5.09/3.92, 6.72/5.49; at 512 rows 3.98/4.52 and 7.92/7.09, at
// 1,024 4.84/6.32 and 13.3/14.3. The activation at 1 / 16 / 256 / 300 / 512 rows of 5,120: 4.16/3.64, 4.47/3.92, 5.34/4.86,
// 5.66/5.72, 5.85/6.24 (the two cross at about 300 rows, the line lies at 512; of 8,192 at 512: 6.99/7.10); of 17,408 at 1 / 16 /
// 512 / 2,048: 7.92/5.55, 8.35/6.02, 14.0/12.4, 35.9/32.6 (5,120 there: 13.5/16.7); of 12,288 at 2,048 / 4,096 rows 25.8/24.6 and
// 42.4/43.3. Rows of 4,096: the two forms are within 4 % up to 256 rows (a thread of either owns one group).
static std::string row_form(const char *base, uint32_t rows, uint32_t width, bool silu = false) {
  if (width <= 2048 && rows % 4 == 0 && rows >= 64) return std::string(base) + "_w64";  // up to two groups a lane
  if (width > T1024_WIDTH_OVER &&
      (silu ? rows <= T1024_SILU_ROWS || width >= T1024_WIDE
            : rows <= (width >= T1024_WIDE ? T1024_QUANT_ROWS_WIDE : T1024_QUANT_ROWS)))
    return std::string(base) + "_t1024";
  const uint32_t slots = (width + 4095) / 4096;
  return std::string(base) + "_t256" + (slots <= 1 ? "_g1" : slots <= 2 ? "_g2" : slots <= 5 ? "_g5" : "");
}

int resolve_quant(uint32_t m, uint32_t k, saber_iu8_desc *out) {
  return describe_rows("quant_i8", row_form("macaq_i8_quant", m, k).c_str(), m, k, "k", out);
}

int resolve_rowscale(uint32_t m, uint32_t k, saber_iu8_desc *out) {
  const uint32_t slots = (k + 4095) / 4096;
  const std::string name = std::string("macaq_i8_rowscale_t256") + (slots <= 1 ? "_g1" : slots <= 2 ? "_g2" : "");
  return describe_rows("rowscale_i8", name.c_str(), m, k, "k", out);
}

// The fused-quant tile GEMM of a shape: the 128 x 128 cell while few tiles would leave CUs idle on the
// larger one, else the 256 x 160 cell (the widest whose registers hold the bf16 pieces in flight).
int resolve_prefill_fused(int wkind, uint32_t m, uint32_t n, uint32_t k, saber_iu8_desc *out) {
  if (wkind != SABER_IU8_W4 && wkind != SABER_IU8_W8) return fail(SABER_IU8_E_ARG, "unknown weight kind");
  const char *tag = wkind == SABER_IU8_W8 ? "w8" : "w4";
  const uint64_t big = (uint64_t)((m + 255) / 256) * ((n + 159) / 160);
  return describe(fmt("macaq_iu8_pfq_%s_%s", tag, big >= CU_COUNT ? "t256x160" : "t128x128"), m, n, k, 1, out);
}

int resolve_quant_rowmajor(uint32_t m, uint32_t k, saber_iu8_desc *out) {
  const uint32_t slots = (k + 4095) / 4096;
  const std::string name = std::string("macaq_i8_quant_rm_t256") + (slots <= 1 ? "_g1" : slots <= 2 ? "_g2" : "");
  return describe_rows("quant_i8_rowmajor", name.c_str(), m, k, "k", out);
}

int resolve_quant_rows(uint32_t rows, uint32_t k, saber_iu8_desc *out) {
  const uint32_t slots = (k + 4095) / 4096;
  const std::string name = std::string("macaq_i8_quant_rows_t256") + (slots <= 1 ? "_g1" : slots <= 2 ? "_g2" : "");
  return describe_rows("quant_rows_i8", name.c_str(), rows, k, "k", out);
}

int resolve_silu_mul_quant(uint32_t rows, uint32_t n, saber_iu8_desc *out) {
  if (int rc = describe_rows("silu_mul_quant_i8", row_form("macaq_i8_silu_mul_quant", rows, n, true).c_str(), rows, n, "n", out)) return rc;
  // the dense form has no row map; the routed form binds both (set_buffer)
  set_null(out, "row_tok");
  set_null(out, "meta");
  return 0;
}

}  // namespace iu8
