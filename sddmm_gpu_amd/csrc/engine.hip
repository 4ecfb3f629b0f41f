// The C entry points of the SDDMM engine for gfx950 (MI355X): plan creation, the execute family,
// values, profiling.  The planner is in planner.hip / planner_tile.hip, plan files in plan_file.hip.
#include <hip/hip_runtime.h>
#include <chrono>
#include <cstring>
#include <new>
#include <unistd.h>
#include "launch.hpp"
#include "plan.hpp"

using namespace sddmm;

extern "C" {

void sddmm_plan_options_init(sddmm_plan_options *opt)
{
    if (opt) default_options(*opt);
}

int sddmm_plan_get_options(const sddmm_plan *plan, sddmm_plan_options *opt)
{
    if (!plan || !opt) return fail(SDDMM_ERR_ARG, "sddmm_plan_get_options: NULL argument");
    *opt = plan->options;
    return SDDMM_OK;
}

int sddmm_plan_create_opt(const sddmm_coo *S, int32_t K, const sddmm_plan_options *opt_in, sddmm_plan **out)
{
    if (!S || !out) return fail(SDDMM_ERR_ARG, "sddmm_plan_create: NULL argument");
    *out = nullptr;
    if (S->sorted != 1) return fail(SDDMM_ERR_UNSORTED, "sddmm_plan_create: matrix is not (row, col)-sorted; call sddmm_coo_sort_rows");
    sddmm_plan_options opt;
    default_options(opt);
    if (opt_in) opt = *opt_in;
    try {
        std::vector<int32_t> rp;
        build_row_ptr(*S, rp);
        return make_plan(S->n_rows, S->n_cols, S->nnz, rp.data(), S->cols.data(), S->vals.data(), nullptr, nullptr, K, opt, out);
    } catch (const std::exception &e) {
        return fail(SDDMM_ERR_NOMEM, "sddmm_plan_create: %s", e.what());
    }
}

int sddmm_plan_create(const sddmm_coo *S, int32_t K, int32_t tile_size_x, int32_t tile_size_y, uint32_t flags,
                      sddmm_plan **out)
{
    sddmm_plan_options opt;
    default_options(opt);
    opt.kernel = (int32_t)(flags & 0xffu); opt.tile_size_x = tile_size_x; opt.tile_size_y = tile_size_y;
    return sddmm_plan_create_opt(S, K, &opt, out);
}

int sddmm_plan_create_device(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *d_row_ptr,
                             const int32_t *d_col_ind, int32_t K, int32_t tile_size_x, int32_t tile_size_y,
                             uint32_t flags, sddmm_plan **out)
{
    sddmm_plan_options opt;
    default_options(opt);
    opt.kernel = (int32_t)(flags & 0xffu); opt.tile_size_x = tile_size_x; opt.tile_size_y = tile_size_y;
    return sddmm_plan_create_device_opt(n_rows, n_cols, nnz, d_row_ptr, d_col_ind, K, &opt, out);
}

int sddmm_plan_create_device_opt(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *d_row_ptr,
                                 const int32_t *d_col_ind, int32_t K, const sddmm_plan_options *opt_in, sddmm_plan **out)
{
    sddmm_plan_options opt;
    default_options(opt);
    if (opt_in) opt = *opt_in;
    if (!out) return fail(SDDMM_ERR_ARG, "sddmm_plan_create_device: out is NULL");
    *out = nullptr;
    if (n_rows < 0 || n_cols < 0 || nnz < 0 || !d_row_ptr || (nnz > 0 && !d_col_ind))
        return fail(SDDMM_ERR_ARG, "sddmm_plan_create_device: bad sizes or NULL arrays");
    if (nnz >= INT32_MAX - 4096 || n_rows >= INT32_MAX || n_cols >= INT32_MAX)
        return fail(SDDMM_ERR_RANGE, "sddmm_plan_create_device: sizes beyond int32 offsets");
    if (int rc = device_ok()) return rc;
    try {
        std::vector<int32_t> rp((size_t)n_rows + 1), ci((size_t)nnz);
        HIP_TRY(hipMemcpy(rp.data(), d_row_ptr, rp.size() * 4, hipMemcpyDeviceToHost));
        if (nnz) HIP_TRY(hipMemcpy(ci.data(), d_col_ind, ci.size() * 4, hipMemcpyDeviceToHost));
        if (rp[0] != 0 || rp[(size_t)n_rows] != nnz)
            return fail(SDDMM_ERR_ARG, "sddmm_plan_create_device: row_ptr does not span [0, nnz]");
        std::vector<char> bad((size_t)hw_threads() + 1, 0);
        parallel_ranges(n_rows, 1 << 12, [&](int64_t b, int64_t e, int t) {
            for (int64_t r = b; r < e; ++r) {
                if (rp[r + 1] < rp[r]) { bad[t] = 1; return; }
                for (int64_t i = rp[r]; i < rp[r + 1]; ++i) {
                    if (ci[i] < 0 || ci[i] >= n_cols) { bad[t] = 2; return; }
                    if (i > rp[r] && ci[i] < ci[i - 1]) { bad[t] = 3; return; }
                }
            }
        });
        for (char c : bad) {
            if (c == 1) return fail(SDDMM_ERR_ARG, "sddmm_plan_create_device: row_ptr is not monotone");
            if (c == 2) return fail(SDDMM_ERR_RANGE, "sddmm_plan_create_device: a column index lies outside the matrix");
            if (c == 3) return fail(SDDMM_ERR_UNSORTED, "sddmm_plan_create_device: columns are not sorted inside a row");
        }
        return make_plan(n_rows, n_cols, nnz, rp.data(), ci.data(), nullptr, d_row_ptr, d_col_ind, K, opt, out);
    } catch (const std::exception &e) {
        return fail(SDDMM_ERR_NOMEM, "sddmm_plan_create_device: %s", e.what());
    }
}

int sddmm_plan_get_info(const sddmm_plan *plan, sddmm_plan_info *info)
{
    if (!plan || !info) return fail(SDDMM_ERR_ARG, "sddmm_plan_get_info: NULL argument");
    *info = plan->info;
    info->device_bytes += plan->host_bytes.load();
    return SDDMM_OK;
}

void sddmm_plan_destroy(sddmm_plan *plan) { delete plan; }

static int check_execute_args(const sddmm_plan *plan, const float *d_W, const float *d_H, float *d_out, const char *who)
{
    if (!plan) return fail(SDDMM_ERR_ARG, "%s: plan is NULL", who);
    if (plan->info.nnz == 0) return SDDMM_OK;
    if (!d_W || !d_H || !d_out) return fail(SDDMM_ERR_ARG, "%s: NULL device pointer", who);
    if ((((uintptr_t)d_W | (uintptr_t)d_H) & 15u) && plan->info.K % 4 == 0)
        return fail(SDDMM_ERR_ARG, "%s: W and H must be 16-byte aligned", who);
    return SDDMM_OK;
}

// A row gather's or an unpadded tile's arguments: what it reads values from and writes to.
static KArgs gather_args(const sddmm_plan *plan, const Launch &L, const float *d_val, float *d_out)
{
    KArgs a = L.ka;
    a.val = d_val ? d_val : plan->d_val;
    a.sval = d_val ? nullptr : L.sval;
    a.out = d_out;
    return a;
}

// Issues the kernels of one launch-list entry (one per K slice) on `stream`.
// ws: the caller's workspace (null: the plan's own scratch memory); softmax: of the rows as well (see softmax_in_launch)
static hipError_t issue_launch(const sddmm_plan *plan, const Launch &L, const float *d_val, const float *d_W,
                         const float *d_H, float *d_out, hipStream_t stream, int epilogue = SDDMM_EPILOGUE_SCALE, char *ws = nullptr, bool softmax = false)
{
    const int residual = epilogue == SDDMM_EPILOGUE_RESIDUAL;
    const sddmm_plan_info &I = plan->info;
    const float *val = d_val ? d_val : plan->d_val;
    if (L.kind == SDDMM_KERNEL_PANEL) {
        PanelArgs pa = L.pa;
        pa.row_ptr = plan->d_row_ptr; pa.col_ind = plan->d_col;
        pa.val = val; pa.W = d_W; pa.H = d_H; pa.out = d_out;
        pa.residual = residual;
        for (int k_off = 0; k_off < I.K; k_off += L.k_slice) {
            pa.k_off = k_off;
            pa.accumulate = k_off > 0;
            if (hipError_t e = launch(L.pfn, dim3((unsigned)L.grid), dim3((unsigned)L.block), (size_t)L.lds, stream, pa)) return e;
        }
        return hipSuccess;
    } else if (L.dfn) {
        DenseArgs da = L.da;
        da.nz_val = d_val ? nullptr : L.sval;
        da.val = val;
        da.W = d_W; da.H = d_H; da.out = d_out;
        da.residual = residual;
        return launch(L.dfn, dim3((unsigned)L.grid), dim3((unsigned)L.block), 0, stream, da);
    } else if (L.bfns[0]) {
        BlockArgs ba = L.ba;
        ba.val = val; ba.W = d_W; ba.H = d_H; ba.out = d_out;
        ba.residual = residual;
        if (!softmax) return launch(L.bfns[0], dim3((unsigned)L.grid), dim3((unsigned)L.block), std::min<size_t>((size_t)L.lds, (size_t)kRoundTiles * kBlockTileBytes), stream, ba);
        if (ws && ba.long_records) ba.long_records = reinterpret_cast<float2 *>(ws + L.ws_part);
        if (hipError_t e = launch(L.bfns[1], dim3((unsigned)L.grid), dim3((unsigned)(64 * L.softmax_waves)), (size_t)L.lds, stream, ba)) return e;
        return launch_block_long_rows(ba, stream);
    } else if (L.tfn) {
        TileArgs ta = L.ta;
        ta.val = val;
        ta.sval = d_val ? nullptr : L.sval;
        ta.W = d_W; ta.H = d_H; ta.out = d_out;
        ta.nnz = (int32_t)I.nnz;
        if (ws) {
            if (ta.part) ta.part = reinterpret_cast<float *>(ws + L.ws_part);
            if (ta.mf_groups > 0) {
                ta.mf_hp = reinterpret_cast<const float4 *>(ws + L.ws_hp);
                ta.mf_wp = reinterpret_cast<const float4 *>(ws + L.ws_wp);
            }
        }
        if (ta.mf_groups > 0) {  // the matrix-core share reads its operands from packed copies of H and of its W rows
            ta.k_off = 0;
            launch_mf_pack(ta, stream);
        }
        const int vm = residual ? (ta.sval ? 3 : 4) : ta.sval ? 0 : (val ? 1 : 2);
        const bool sliced = L.k_slice < I.K;
        if (sliced && L.fused_slices) {
            ta.k_off = 0; ta.n_slices = (I.K + L.k_slice - 1) / L.k_slice;
            return launch(L.tfns[vm][3], dim3((unsigned)L.grid), dim3((unsigned)L.block), (size_t)L.lds, stream, ta);
        }
        for (int k_off = 0; k_off < I.K; k_off += L.k_slice) {
            ta.k_off = k_off;
            const int slice = !sliced ? 0 : k_off + L.k_slice >= I.K ? 4 : k_off == 0 ? 1 : 2;
            if (hipError_t e = launch(L.tfns[vm][slice], dim3((unsigned)L.grid), dim3((unsigned)L.block), (size_t)L.lds,
                                      stream, ta))
                return e;
        }
        return hipSuccess;
    } else {
        KArgs a = gather_args(plan, L, d_val, d_out);
        a.col_ind = plan->d_col;
        a.W = d_W; a.H = d_H;
        a.residual = residual;
        if (L.fn_kind == 1 && L.k_slice < I.K) return launch_gather_slices(a, L.rows, I.n_rows, L.fn_wide != 0, L.k_slice, stream);
        return launch(L.fn, dim3((unsigned)L.grid), dim3((unsigned)L.block), (size_t)L.lds, stream, a);
    }
}

// Row blocks take the softmax along, without a pass over out.  (Rows whose blocks are several units get a pass of their own, a
// workgroup per 16,384 entries: where they are many the general pass is the faster one.)
static bool softmax_in_launch(const sddmm_plan *plan)
{
    return plan->launches.size() == 1 && plan->launches[0].bfns[1] && plan->launches[0].ba.n_long_pieces <= 1024;
}

int sddmm_execute(const sddmm_plan *plan, const float *d_val, const float *d_W, const float *d_H, float *d_out,
                  void *stream)
{
    if (int rc = check_execute_args(plan, d_W, d_H, d_out, "sddmm_execute")) return rc;
    if (plan->info.nnz == 0) return SDDMM_OK;
    for (const Launch &L : plan->launches) HIP_TRY(issue_launch(plan, L, d_val, d_W, d_H, d_out, (hipStream_t)stream));
    return SDDMM_OK;
}

int sddmm_execute_epilogue(const sddmm_plan *plan, const float *d_val, const float *d_W, const float *d_H, float *d_out,
                           int32_t epilogue, void *stream)
{
    if (int rc = check_execute_args(plan, d_W, d_H, d_out, "sddmm_execute_epilogue")) return rc;
    if (epilogue != SDDMM_EPILOGUE_SCALE && epilogue != SDDMM_EPILOGUE_RESIDUAL)
        return fail(SDDMM_ERR_ARG, "sddmm_execute_epilogue: unknown epilogue %d", (int)epilogue);
    if (epilogue == SDDMM_EPILOGUE_RESIDUAL && !d_val && !plan->d_val && plan->info.nnz > 0)
        return fail(SDDMM_ERR_ARG, "sddmm_execute_epilogue: the residual val - dot needs values (d_val or plan-owned)");
    if (plan->info.nnz == 0) return SDDMM_OK;
    for (const Launch &L : plan->launches) HIP_TRY(issue_launch(plan, L, d_val, d_W, d_H, d_out, (hipStream_t)stream, epilogue));
    return SDDMM_OK;
}

int sddmm_execute_softmax(const sddmm_plan *plan, const float *d_val, const float *d_W, const float *d_H, float *d_out,
                          void *stream)
{
    if (int rc = check_execute_args(plan, d_W, d_H, d_out, "sddmm_execute_softmax")) return rc;
    if (plan->info.nnz == 0) return SDDMM_OK;
    const bool in_launch = softmax_in_launch(plan);
    for (const Launch &L : plan->launches)
        HIP_TRY(issue_launch(plan, L, d_val, d_W, d_H, d_out, (hipStream_t)stream, SDDMM_EPILOGUE_SCALE, nullptr, in_launch));
    if (in_launch) return SDDMM_OK;
    if (!plan->d_row_ptr) return fail(SDDMM_ERR_ARG, "sddmm_execute_softmax: the plan holds no row pointers");
    return launch_row_softmax(plan->info.n_rows, plan->d_row_ptr, d_out, d_out, stream, nullptr, 0, plan->launches[0].longest_row);
}

int sddmm_plan_workspace_bytes(const sddmm_plan *plan, int64_t *bytes)
{
    if (!plan || !bytes) return fail(SDDMM_ERR_ARG, "sddmm_plan_workspace_bytes: NULL argument");
    *bytes = plan->ws_bytes;
    return SDDMM_OK;
}

int sddmm_execute_ws(const sddmm_plan *plan, const float *d_val, const float *d_W, const float *d_H, float *d_out,
                     int32_t form, void *d_workspace, int64_t workspace_bytes, void *stream)
{
    if (int rc = check_execute_args(plan, d_W, d_H, d_out, "sddmm_execute_ws")) return rc;
    const int32_t epilogue = form & 0xff;
    const bool softmax = (form & SDDMM_FORM_SOFTMAX) != 0;
    if ((form & ~(0xff | SDDMM_FORM_SOFTMAX)) || (epilogue != SDDMM_EPILOGUE_SCALE && epilogue != SDDMM_EPILOGUE_RESIDUAL))
        return fail(SDDMM_ERR_ARG, "sddmm_execute_ws: unknown form %d", (int)form);
    if (epilogue == SDDMM_EPILOGUE_RESIDUAL && !d_val && !plan->d_val && plan->info.nnz > 0)
        return fail(SDDMM_ERR_ARG, "sddmm_execute_ws: the residual val - dot needs values (d_val or plan-owned)");
    if (plan->info.nnz == 0) return SDDMM_OK;
    if (plan->ws_bytes > 0 && (!d_workspace || workspace_bytes < plan->ws_bytes))
        return fail(SDDMM_ERR_ARG, "sddmm_execute_ws: the plan needs a workspace of %lld bytes (sddmm_plan_workspace_bytes)",
                    (long long)plan->ws_bytes);
    if ((uintptr_t)d_workspace & 255u) return fail(SDDMM_ERR_ARG, "sddmm_execute_ws: the workspace must be 256-byte aligned");
    char *ws = static_cast<char *>(d_workspace);
    const bool in_launch = softmax && softmax_in_launch(plan);
    for (const Launch &L : plan->launches) HIP_TRY(issue_launch(plan, L, d_val, d_W, d_H, d_out, (hipStream_t)stream, epilogue, ws, in_launch));
    if (!softmax || in_launch) return SDDMM_OK;
    if (!plan->d_row_ptr) return fail(SDDMM_ERR_ARG, "sddmm_execute_ws: the plan holds no row pointers");
    return launch_row_softmax(plan->info.n_rows, plan->d_row_ptr, d_out, d_out, stream, ws + plan->ws_softmax, plan->info.nnz, plan->launches[0].longest_row);
}

static const Launch *spmm_launch(const sddmm_plan *plan)
{
    const Launch *found = nullptr;
    for (const Launch &L : plan->launches)
        if (L.sp_on) found = &L;
    return found;
}

int sddmm_plan_spmm_form(const sddmm_plan *plan, int32_t *form)
{
    if (!plan || !form) return fail(SDDMM_ERR_ARG, "sddmm_plan_spmm_form: NULL argument");
    const Launch *L = spmm_launch(plan);
    *form = !L ? SDDMM_SPMM_CSR : L->sp_on == 1 ? SDDMM_SPMM_TILES : L->sp_on == 2 ? SDDMM_SPMM_WALK : SDDMM_SPMM_BLOCKS;
    return SDDMM_OK;
}

int sddmm_plan_spmm(const sddmm_plan *plan, const float *d_x, const float *d_H, float *d_Y, void *d_workspace,
                    int64_t workspace_bytes, void *stream)
{
    if (!plan) return fail(SDDMM_ERR_ARG, "sddmm_plan_spmm: plan is NULL");
    const sddmm_plan_info &I = plan->info;
    if (I.n_rows == 0) return SDDMM_OK;
    if (!d_Y || (I.nnz > 0 && (!d_x || !d_H))) return fail(SDDMM_ERR_ARG, "sddmm_plan_spmm: NULL device pointer");
    const Launch *Ls = spmm_launch(plan);
    if (!Ls || (Ls->sp_on == 1 && !Ls->fn_ragged && ((((uintptr_t)d_H) | ((uintptr_t)d_Y)) & 15u))) {
        // no tile stream for the product in this plan: the CSR form, gathering H rows
        if (!plan->d_row_ptr || (I.nnz > 0 && !plan->d_col)) return fail(SDDMM_ERR_ARG, "sddmm_plan_spmm: the plan holds no pattern");
        return sddmm_spmm_csr(I.n_rows, I.n_cols, I.nnz, plan->d_row_ptr, plan->d_col, d_x, I.K, d_H, d_Y, stream);
    }
    if (d_workspace) {
        if (workspace_bytes < plan->ws_bytes) return fail(SDDMM_ERR_ARG, "sddmm_plan_spmm: the plan needs a workspace of %lld bytes", (long long)plan->ws_bytes);
        if ((uintptr_t)d_workspace & 255u) return fail(SDDMM_ERR_ARG, "sddmm_plan_spmm: the workspace must be 256-byte aligned");
    }
    if (Ls->sp_on == 2)
        return launch_spmm_csr_records(I.n_rows, I.n_cols, I.nnz, plan->d_row_ptr, plan->d_col, d_x, I.K, d_H, d_Y,
                                       d_workspace ? reinterpret_cast<float *>(static_cast<char *>(d_workspace) + Ls->ws_sp_part) : Ls->sa.part, stream);
    if (Ls->sp_on == 3) {
        BlockArgs ba = Ls->ba;
        ba.x = d_x; ba.H = d_H; ba.Y = d_Y;
        if (d_workspace) ba.part = reinterpret_cast<float *>(static_cast<char *>(d_workspace) + Ls->ws_sp_part);
        HIP_TRY(launch_block_spmm(ba, Ls->fn_nwaves, stream));
        return SDDMM_OK;
    }
    SpmmArgs sa = Ls->sa;
    sa.x = d_x; sa.H = d_H; sa.Y = d_Y;
    sa.row_ptr = plan->d_row_ptr; sa.col_ind = plan->d_col;
    if (d_workspace) sa.part = reinterpret_cast<float *>(static_cast<char *>(d_workspace) + Ls->ws_sp_part);
    const int width = 4 * Ls->fn_g * Ls->fn_kpl;  // (k_slice is K where a wider kernel covers a ragged rank)
    for (int k_off = 0; k_off < I.K; k_off += width) {
        sa.k_off = k_off;
        launch_spmm_slice(sa, width, Ls->sp_nwaves, Ls->sp_grid, width * 4 * Ls->ta.tile_x, stream);
    }
    HIP_TRY(hipGetLastError());
    return SDDMM_OK;
}

int sddmm_plan_set_values(sddmm_plan *plan, const float *d_val, void *stream)
{
    if (!plan) return fail(SDDMM_ERR_ARG, "sddmm_plan_set_values: plan is NULL");
    const int64_t nnz = plan->info.nnz;
    if (nnz == 0) return SDDMM_OK;
    if (!d_val) return fail(SDDMM_ERR_ARG, "sddmm_plan_set_values: d_val is NULL");
    if (!plan->d_val) {
        HIP_TRY(hipMalloc((void **)&plan->d_val, (size_t)nnz * 4));
        plan->owned.push_back({plan->d_val, (size_t)nnz * 4});
        plan->info.device_bytes += nnz * 4;
    }
    HIP_TRY(hipMemcpyAsync(plan->d_val, d_val, (size_t)nnz * 4, hipMemcpyDeviceToDevice, (hipStream_t)stream));
    for (Launch &L : plan->launches) {
        if (!L.perm || L.positions <= 0) continue;  // walks S in sorted order: reads d_val directly
        if (!L.sval) {
            HIP_TRY(hipMalloc((void **)&L.sval, ((size_t)L.positions + kStreamSlack) * 4));  // (see add_tile)
            plan->owned.push_back({L.sval, ((size_t)L.positions + kStreamSlack) * 4});
            plan->info.device_bytes += L.positions * 4;
        }
        launch_gather_values(L.perm, plan->d_val, L.sval, L.positions, stream);
    }
    HIP_TRY(hipGetLastError());
    return SDDMM_OK;
}

int sddmm_plan_launch_count(const sddmm_plan *plan, int32_t *n)
{
    if (!plan || !n) return fail(SDDMM_ERR_ARG, "sddmm_plan_launch_count: NULL argument");
    *n = (int32_t)plan->launches.size();
    return SDDMM_OK;
}

int sddmm_execute_profiled(const sddmm_plan *plan, const float *d_val, const float *d_W, const float *d_H,
                           float *d_out, void *stream, sddmm_launch_profile *prof, int32_t max_prof)
{
    if (int rc = check_execute_args(plan, d_W, d_H, d_out, "sddmm_execute_profiled")) return rc;
    if (!prof || max_prof < (int32_t)plan->launches.size())
        return fail(SDDMM_ERR_ARG, "sddmm_execute_profiled: room for %zu profiles needed", plan->launches.size());
    if (plan->info.nnz == 0) return SDDMM_OK;
    const size_t n = plan->launches.size();
    std::vector<hipEvent_t> ev(n + 1, nullptr);
    struct Ev { std::vector<hipEvent_t> &e; ~Ev() { for (auto x : e) if (x) (void)hipEventDestroy(x); } } guard{ev};
    for (auto &x : ev) HIP_TRY(hipEventCreate(&x));
    HIP_TRY(hipEventRecord(ev[0], (hipStream_t)stream));
    for (size_t i = 0; i < n; ++i) {
        HIP_TRY(issue_launch(plan, plan->launches[i], d_val, d_W, d_H, d_out, (hipStream_t)stream));
        HIP_TRY(hipEventRecord(ev[i + 1], (hipStream_t)stream));
    }
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipEventSynchronize(ev[n]));
    for (size_t i = 0; i < n; ++i) {
        const Launch &L = plan->launches[i];
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, ev[i], ev[i + 1]));
        prof[i].kernel = L.kind;
        prof[i].lanes_per_nnz = L.dfn || L.bfns[0] ? 0 : L.kind == SDDMM_KERNEL_PANEL ? 8 : (L.tfn ? L.tile_g : L.gather_g);
        prof[i].k_slice = L.k_slice;
        const bool slices = L.k_slice > 0 && L.k_slice < plan->info.K && !L.fused_slices;
        prof[i].n_kernel_launches = !slices ? 1 : L.fn_kind == 1 ? gather_slice_launches(gather_args(plan, L, d_val, d_out), L.k_slice)
                                                                 : (plan->info.K + L.k_slice - 1) / L.k_slice;
        prof[i].nnz = L.nnz;
        prof[i].rows = L.rows;
        prof[i].stream_positions = L.positions;
        prof[i].ms = ms;
    }
    return SDDMM_OK;
}

int sddmm_device_info(int *n_devices, char *arch, int arch_len)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
    if (n_devices) *n_devices = n;
    if (arch && arch_len > 0) {
        arch[0] = 0;
        if (n > 0) {
            hipDeviceProp_t prop;
            if (hipGetDeviceProperties(&prop, 0) == hipSuccess) {
                strncpy(arch, prop.gcnArchName, (size_t)arch_len - 1);
                arch[arch_len - 1] = 0;
            }
        }
    }
    return SDDMM_OK;
}

}  // extern "C"
