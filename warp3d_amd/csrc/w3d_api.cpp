// w3d_api.cpp -- the C ABI of libw3dblk (include/w3d.h): model set-up,
// blocking, device state, orchestration of the kernels, sparsity pattern and
// the host views of block state.
//
// Reference set-up steps restated here (file:line under the reference's
// src/): inelbk.f:282-548 automatic blocking and its compatibility rules,
// setup.f:160-190 inverse incidences, reopen.f:1315 edest_init,
// elprp.f:872 H' = E Et / (E - Et) in REAL, rknstr.f:1018
// setup_mm01_rknstr, assemble_code.f:561 dof_map, :20 / :260
// count_profile_symmetric / build_col_sparse_symm, update.f:15.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "w3d_ctx.h"

namespace w3d {
bool fill_gauss_table(int etype, int order, GaussTable* t);
int ngp_of(int etype, int order);
int nnode_of(int etype);
}  // namespace w3d

using namespace w3d;

namespace {
thread_local std::string g_err = "no error";
}  // namespace

thread_local int64_t w3d::t_dalloc_bytes = 0;

int w3d::fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

namespace {

// H' = E Et / (E - Et) in single precision
float hprime_real(float e, float et) {
  volatile float num = e * et;  // REAL arithmetic as elprp.f:872
  volatile float den = e - et;
  return num / den;
}

}  // namespace


namespace w3d {

bool compatible(const w3d_ctx* c, int a, int b) {
  return c->etype[a] == c->etype[b] && c->matnum[a] == c->matnum[b] &&
         c->order[a] == c->order[b] &&
         ngp_of(c->etype[a], c->order[a]) == ngp_of(c->etype[b], c->order[b]) &&
         c->bbar[a] == c->bbar[b] && c->geonl[a] == c->geonl[b];
}

// inelbk_simple_blocking (inelbk.f:282): one sequential pass; a new block
// opens when the current one is full or the element is incompatible with
// the block's first element.
void auto_blocking(w3d_ctx* c, int auto_size) {
  c->elblks.assign({1, 1, 0, 0});
  int nb = 1, cur = 1, felem = 1;
  for (int e = 2; e <= c->noelem; ++e) {
    bool newblk = false;
    cur = cur + 1;
    if (cur > auto_size) newblk = true;
    if (!newblk && !compatible(c, felem - 1, e - 1)) newblk = true;
    if (!newblk) {
      c->elblks[4 * (nb - 1)] = cur;
      continue;
    }
    nb += 1;
    felem = e;
    c->elblks.insert(c->elblks.end(), {1, felem, 0, 0});
    cur = 1;
  }
  c->nelblk = nb;
}

// Work lists: chunks of consecutive elements of one block, grouped by
// kernel instantiation.
void build_work(const w3d_ctx* c, bool tangent, std::vector<WorkItem>& items,
                std::vector<int>& groups, std::vector<int>& start,
                std::vector<int>& count) {
  std::vector<std::pair<int, WorkItem>> all;
  auto key_of = [&](const BlockDesc& B) {
    return group_key(B.nnode, B.ngp, B.bbar,
                     !tangent && B.model == W3D_MM10, B.geonl,
                     tangent && B.trn);
  };
  std::map<int, int64_t> nelem;  // elements of each kernel group
  for (const BlockDesc& B : c->blocks) nelem[key_of(B)] += B.span;
  for (int b = 0; b < c->nelblk; ++b) {
    const BlockDesc& B = c->blocks[b];
    const int key = key_of(B);
    int E = tangent ? tan_mfma_chunk(B.nnode) : rec_elems(B.ngp);
    if (tangent) {
      // a group of less than three workgroups on two compute units takes
      // smaller items, down to an element a wave (tangent of 1,000 bricks,
      // FP64: 26.3 us in items of 32, 15.3 of 16, 9.7 of 4; of 10,296
      // tetrahedra 28.1 us of 32, 22.3 of 16, 26.5 of 8); larger groups lose
      // by it (14,400 bricks, FP32: 29.3 us of 32, 33.9 of 16)
      while (E > tan_mfma_waves(B.nnode) && nelem[key] / E < 3 * c->n_cu / 2)
        E /= 2;
      for (const auto& kc : c->tan_chunk)
        if (kc.first == key) E = kc.second;
    }
    for (int f = 0; f < B.span; f += E) {
      WorkItem w;
      w.blk = b;
      w.first = f;
      w.count = std::min(E, B.span - f);
      w.pad_ = 0;
      all.push_back({key, w});
    }
  }
  std::stable_sort(all.begin(), all.end(),
                   [](const auto& x, const auto& y) { return x.first < y.first; });
  items.clear();
  groups.clear();
  start.clear();
  count.clear();
  for (size_t k = 0; k < all.size(); ++k) {
    if (groups.empty() || groups.back() != all[k].first) {
      groups.push_back(all[k].first);
      start.push_back((int)k);
      count.push_back(0);
    }
    count.back() += 1;
    items.push_back(all[k].second);
  }
}

// Each block's run of items in the recovery and tangent work lists (a
// block's items are consecutive inside its kernel group) and in the mm10
// list, for the per-block calls.
void build_runs(w3d_ctx* c) {
  c->runs.assign(c->nelblk, w3d_ctx::BlockRuns());
  for (int pass = 0; pass < 2; ++pass) {
    std::vector<WorkItem> items;
    std::vector<int> g, st, n;
    build_work(c, pass == 1, items, g, st, n);
    for (size_t k = 0; k < g.size(); ++k)
      for (int i = st[k]; i < st[k] + n[k]; ++i) {
        w3d_ctx::BlockRuns& R = c->runs[items[i].blk];
        int &key = pass ? R.tan_key : R.rec_key;
        int &first = pass ? R.tan_first : R.rec_first;
        int &cnt = pass ? R.tan_n : R.rec_n;
        if (cnt == 0) {
          key = g[k];
          first = i;
        }
        cnt += 1;
      }
  }
  int item = 0, idx = 0;
  for (int b = 0; b < c->nelblk; ++b) {
    const BlockDesc& B = c->blocks[b];
    if (B.model != W3D_MM10) continue;
    const int np = B.span * B.ngp;
    c->runs[b].mm10_first = item;
    c->runs[b].mm10_n = (np + 63) / 64;   // items of 64 points (w3d_create)
    c->runs[b].mm10_idx = idx++;
    item += c->runs[b].mm10_n;
  }
}

// A context's pinned image: a solve's scalars and states (8 words), then
// what a recovery leaves for the host (launch_recover_end).
size_t pin_words(const w3d_ctx* c) {
  return 8 + kBlkSums * (size_t)c->nelblk + 2;
}

void free_ctx(w3d_ctx* c) {
  dfree(c->d_blocks); dfree(c->d_mats); dfree(c->d_tables);
  dfree(c->d_coords); dfree(c->d_conn);
  dfree(c->d_stress_n); dfree(c->d_stress_n1);
  dfree(c->d_strain_n); dfree(c->d_strain_n1);
  dfree(c->d_hist_n); dfree(c->d_hist_n1); dfree(c->d_cep);
  dfree(c->d_ek64); dfree(c->d_ek32); dfree(c->d_einfvec);
  dfree(c->d_evol); dfree(c->d_en_wg); dfree(c->d_flags);
  dfree(c->d_work_rec); dfree(c->d_work_tan);
  dfree(c->d_inv_ptr); dfree(c->d_inv_off);
  dfree(c->d_blk_wfirst); dfree(c->d_blk_wcount);
  dfree(c->d_blk_sums); dfree(c->d_u); dfree(c->d_du); dfree(c->d_ifv);
  dfree(c->d_asm_hdr); dfree(c->d_asm_src); dfree(c->d_asm_wbase); dfree(c->d_kout);
  dfree(c->d_csr_rp); dfree(c->d_csr_col); dfree(c->d_csr_vidx);
  dfree(c->d_csr_grp);
  dfree(c->d_csr_val); dfree(c->d_pcg); dfree(c->d_bicg);
  dfree(c->d_ekf); dfree(c->d_ekf_off);
  dfree(c->d_fa_eqdof); dfree(c->d_fa_ln); dfree(c->d_fa_invptr);
  dfree(c->d_fa_ebase); dfree(c->d_fa_atoff); dfree(c->d_fa_at);
  dfree(c->d_crys); dfree(c->d_uddt); dfree(c->d_rot_tmp); dfree(c->d_jac_tmp); dfree(c->d_work_mm10); dfree(c->d_mm10_blks);
  dfree(c->d_rot_n); dfree(c->d_rot_n1); dfree(c->d_u_t); dfree(c->d_du_t);
  dfree(c->d_counter);
  dfree(c->d_blk_flags); dfree(c->d_blk_counter);
  dfree(c->d_trn_idx); dfree(c->d_trn_mat);
  dfree(c->d_therm); dfree(c->d_temps);
  for (hipStream_t st : c->pool_all) (void)hipStreamDestroy(st);
  c->pool_all.clear();
  c->pool_idle.clear();
  for (auto& g : c->graphs) (void)hipGraphExecDestroy(g.exec);
  c->graphs.clear();
  for (int ph = 0; ph < W3D_NUM_PHASES; ++ph) {
    for (int k = 0; k < 2; ++k) {
      if (c->ev_a[ph][k]) hipEventDestroy(c->ev_a[ph][k]);
      if (c->ev_b[ph][k]) hipEventDestroy(c->ev_b[ph][k]);
      c->ev_a[ph][k] = c->ev_b[ph][k] = nullptr;
    }
  }
  for (int k = 0; k < 2; ++k) {
    if (c->poll_ev[k]) (void)hipEventDestroy(c->poll_ev[k]);
    c->poll_ev[k] = nullptr;
    c->h_poll[k] = nullptr;
  }
  if (c->h_poll_sc) (void)hipHostFree(c->h_poll_sc);
  c->h_poll_sc = c->h_rec = nullptr;
  if (c->stream) hipStreamDestroy(c->stream);
  c->stream = nullptr;
}


int create_impl(w3d_ctx* c, const w3d_model* m) {
  if (m->nonode <= 0 || m->noelem <= 0 || !m->c || !m->incid ||
      !m->incmap || !m->etype || !m->int_order || !m->matnum || !m->mats ||
      m->nmat <= 0)
    return fail(W3D_ERR_ARG, "w3d_create: incomplete model");
  c->nonode = m->nonode;
  c->noelem = m->noelem;
  c->eps_bbar = m->eps_bbar;
  c->etype.resize(m->noelem);
  c->order.resize(m->noelem);
  c->matnum.resize(m->noelem);
  c->bbar.resize(m->noelem);
  c->geonl.resize(m->noelem);
  for (int e = 0; e < m->noelem; ++e) {
    c->geonl[e] = m->geonl && m->geonl[e] ? 1 : 0;
    c->has_geonl = c->has_geonl || c->geonl[e];
    c->etype[e] = m->etype[e];
    c->order[e] = m->int_order[e];
    c->matnum[e] = m->matnum[e];
    c->bbar[e] = m->etype[e] == W3D_L3DISOP && m->bbar && m->bbar[e];
    if (nnode_of(m->etype[e]) == 0 || ngp_of(m->etype[e], m->int_order[e]) == 0)
      return fail(W3D_ERR_UNSUPPORTED,
                  "w3d_create: element type / integration order of element " +
                      std::to_string(e + 1));
    if (m->matnum[e] < 1 || m->matnum[e] > m->nmat)
      return fail(W3D_ERR_ARG, "w3d_create: material number of element " +
                                   std::to_string(e + 1));
  }
  // materials (setup_mm01_rknstr: REAL props widened to FP64)
  c->mats.resize(m->nmat);
  c->therm.resize(m->nmat);
  for (int k = 0; k < m->nmat; ++k) {
    const w3d_material& s = m->mats[k];
    MatDesc& d = c->mats[k];
    std::memset(&d, 0, sizeof d);
    d.model = s.model;
    // thermal expansion (props 9, 13, 34-37, matprp 250) and the segmental
    // curve set
    w3d::ThermDesc& td = c->therm[k];
    std::memset(&td, 0, sizeof td);
    for (int j = 0; j < 6; ++j) td.alpha[j] = (double)s.alpha[j];
    td.alpha_zero = (double)s.alpha_zero;
    td.curve_type = s.curve_type;
    if (s.curve_type != 0) {
      const int nc = s.curve_type == 1 ? 1 : s.ncurves;
      bool ok = s.model == W3D_MM01 &&
                (s.curve_type == 1 || s.curve_type == 2) && nc >= 1 &&
                nc <= w3d::kMaxCurves &&
                s.curve_eps[1] != s.curve_eps[0];
      for (int j = 1; ok && s.curve_type == 2 && j < nc; ++j)
        ok = s.curve_temp[j] > s.curve_temp[j - 1];
      if (!ok)
        return fail(W3D_ERR_ARG, "w3d_create: segmental curves of material " +
                                     std::to_string(k + 1));
      td.ncurves = nc;
      td.curve_eps[0] = s.curve_eps[0];
      td.curve_eps[1] = s.curve_eps[1];
      for (int j = 0; j < nc; ++j) {
        td.temp[j] = s.curve_temp[j];
        td.e[j] = s.curve_e[j];
        td.nu[j] = s.curve_nu[j];
        td.alpha_c[j] = s.curve_alpha[j];
        td.sig[j][0] = s.curve_sig[j][0];
        td.sig[j][1] = s.curve_sig[j][1];
      }
      c->curves = true;
    }
    if (s.model == W3D_MM01) {
      if (!(s.e > s.tan_e) || s.e <= 0.0f || s.nu <= -1.0f || s.nu >= 0.5f)
        return fail(W3D_ERR_ARG, "w3d_create: mm01 properties of material " +
                                     std::to_string(k + 1));
      d.lnelas = s.linear_elastic;
      d.e = (double)s.e;
      d.nu = (double)s.nu;
      d.beta = (double)s.beta;
      d.hprime = (double)hprime_real(s.e, s.tan_e);
      d.yld = (double)s.yld_pt;
    } else if (s.model == W3D_MM10) {
      // the implemented scope: Voce hardening, Kocks angles, 12-system
      // fcc / bcc crystals with isotropic or cubic elasticity
      if ((s.slip_type != 1 && s.slip_type != 2) ||
          (s.elastic_type != 1 && s.elastic_type != 2) ||
          s.angle_convention != 1 ||
          (s.angle_type != 1 && s.angle_type != 2) || s.ncrystals < 1 ||
          s.ncrystals > (m->angle_stride > 0 ? m->angle_stride : 1) ||
          !(s.cp_e > 0.0) || !(s.tau_v > 0.0) || !(s.harden_n > 0.0) ||
          s.miter < 1 || !m->angles)
        return fail(W3D_ERR_UNSUPPORTED,
                    "w3d_create: mm10 properties of material " +
                        std::to_string(k + 1));
      CpDesc& cp = d.cp;
      cp.rate_n = s.harden_n;
      cp.tau_y = s.tau_y;
      cp.tau_v = s.tau_v;
      cp.voce_m = s.voce_m;
      cp.theta_0 = s.theta_0;
      cp.iD_v = s.iD_v;
      cp.eps_dot_0_y = s.eps_dot_0_y;
      cp.atol = s.atol;
      cp.atol1 = s.atol1;
      cp.rtol = s.rtol;
      cp.rtol1 = s.rtol1;
      cp.miter = s.miter;
      cp.alter_mode = s.alter_mode;
      cp.angle_type = s.angle_type;
      cp.ncry = s.ncrystals;
    } else {
      return fail(W3D_ERR_UNSUPPORTED,
                  "w3d_create: material model " + std::to_string(s.model) +
                      " of material " + std::to_string(k + 1));
    }
  }
  // blocking
  if (m->nelblk > 0) {
    if (!m->elblks) return fail(W3D_ERR_ARG, "w3d_create: elblks missing");
    c->nelblk = m->nelblk;
    c->elblks.assign(m->elblks, m->elblks + 4 * m->nelblk);
    int next = 1;
    for (int b = 0; b < c->nelblk; ++b) {
      int span = c->elblks[4 * b], felem = c->elblks[4 * b + 1];
      if (span < 1 || felem != next)
        return fail(W3D_ERR_ARG, "w3d_create: blocks must tile the elements");
      for (int i = 1; i < span; ++i)
        if (!compatible(c, felem - 1, felem - 1 + i))
          return fail(W3D_ERR_ARG,
                      "w3d_create: incompatible elements in block " +
                          std::to_string(b + 1));
      next = felem + span;
    }
    if (next != c->noelem + 1)
      return fail(W3D_ERR_ARG, "w3d_create: blocks must tile the elements");
  } else {
    auto_blocking(c, m->auto_size > 0 ? m->auto_size : 128);
  }
  // Gauss tables
  std::vector<std::pair<int, int>> tkeys;
  auto table_of = [&](int et, int ord) {
    for (size_t k = 0; k < tkeys.size(); ++k)
      if (tkeys[k].first == et && tkeys[k].second == ord) return (int)k;
    tkeys.push_back({et, ord});
    GaussTable t;
    fill_gauss_table(et, ord, &t);
    c->tables.push_back(t);
    return (int)tkeys.size() - 1;
  };
  // blocks
  c->blocks.resize(c->nelblk);
  c->elem_blk.resize(c->noelem);
  int64_t q = 0, h = 0, ek = 0, fv = 0, cn = 0, ncr = 0;
  for (int b = 0; b < c->nelblk; ++b) {
    BlockDesc& B = c->blocks[b];
    std::memset(&B, 0, sizeof B);
    B.span = c->elblks[4 * b];
    B.felem = c->elblks[4 * b + 1];
    int fe = B.felem - 1;
    B.etype = c->etype[fe];
    B.order = c->order[fe];
    B.ngp = ngp_of(B.etype, B.order);
    B.nnode = nnode_of(B.etype);
    B.totdof = 3 * B.nnode;
    B.utsz = B.totdof * (B.totdof + 1) / 2;
    B.mat = c->matnum[fe] - 1;
    B.model = c->mats[B.mat].model;
    B.ncry = B.model == W3D_MM10 ? c->mats[B.mat].cp.ncry : 0;
    B.hist = B.model == W3D_MM01 ? kMM01Hist
                                 : kMM10Common + kMM10Crystal * B.ncry;
    B.bbar = c->bbar[fe];
    B.geonl = c->geonl[fe];
    B.table = table_of(B.etype, B.order);
    B.q_off = q;
    B.hist_off = h;
    B.ek_off = ek;
    B.ifv_off = fv;
    B.conn_off = cn;
    B.crys_off = ncr;
    ncr += (int64_t)B.span * B.ncry;
    q += (int64_t)B.span * B.ngp;
    h += (int64_t)B.span * B.ngp * B.hist;
    ek += (int64_t)B.span * B.utsz;
    fv += (int64_t)B.span * B.totdof;
    cn += (int64_t)B.span * B.nnode;
    for (int i = 0; i < B.span; ++i) c->elem_blk[fe + i] = b;
  }
  c->nq = q;
  c->nhist = h;
  c->nek = ek;
  c->nifv = fv;
  if (ek >= (int64_t)UINT32_MAX)
    return fail(W3D_ERR_UNSUPPORTED, "w3d_create: too many Ke words");
  c->conn.resize(cn);
  for (int b = 0; b < c->nelblk; ++b) {
    const BlockDesc& B = c->blocks[b];
    for (int i = 0; i < B.span; ++i) {
      int e = B.felem - 1 + i;
      for (int j = 0; j < B.nnode; ++j) {
        int node = m->incid[m->incmap[e] - 1 + j];
        if (node < 1 || node > c->nonode)
          return fail(W3D_ERR_ARG, "w3d_create: bad node in element " +
                                       std::to_string(e + 1));
        c->conn[B.conn_off + (int64_t)i * B.nnode + j] = node - 1;
      }
    }
  }
  // skewed constraints (duptrans, tanstf.f:733): node -> matrix index
  if (m->trn && m->trnmat) {
    c->trn_idx.assign(c->nonode, -1);
    for (int n = 0; n < c->nonode; ++n)
      if (m->trn[n]) {
        c->trn_idx[n] = (int32_t)(c->trn_mat.size() / 9);
        c->trn_mat.insert(c->trn_mat.end(), m->trnmat + 9 * (int64_t)n,
                          m->trnmat + 9 * (int64_t)n + 9);
      }
    for (int b = 0; b < c->nelblk; ++b) {
      BlockDesc& B = c->blocks[b];
      for (int64_t k = 0; k < (int64_t)B.span * B.nnode && !B.trn; ++k)
        B.trn = c->trn_idx[c->conn[B.conn_off + k]] >= 0 ? 1 : 0;
    }
    if (c->trn_mat.empty()) c->trn_idx.clear();
  }
  // inverse incidences (element order; repeated nodes listed once)
  c->inv_ptr.assign(c->nonode + 1, 0);
  for (int b = 0; b < c->nelblk; ++b) {
    const BlockDesc& B = c->blocks[b];
    for (int i = 0; i < B.span; ++i) {
      const int32_t* nd = &c->conn[B.conn_off + (int64_t)i * B.nnode];
      for (int j = 0; j < B.nnode; ++j) {
        bool rep = false;
        for (int k = 0; k < j; ++k) rep |= nd[k] == nd[j];
        if (rep)
          return fail(W3D_ERR_UNSUPPORTED,
                      "w3d_create: repeated nodes in an element");
        c->inv_ptr[nd[j] + 1] += 1;
      }
    }
  }
  for (int n = 0; n < c->nonode; ++n) c->inv_ptr[n + 1] += c->inv_ptr[n];
  c->inv_elem.resize(c->inv_ptr[c->nonode]);
  c->inv_ln.resize(c->inv_ptr[c->nonode]);
  {
    std::vector<int64_t> fill(c->inv_ptr.begin(), c->inv_ptr.end() - 1);
    for (int b = 0; b < c->nelblk; ++b) {
      const BlockDesc& B = c->blocks[b];
      for (int i = 0; i < B.span; ++i) {
        const int32_t* nd = &c->conn[B.conn_off + (int64_t)i * B.nnode];
        for (int j = 0; j < B.nnode; ++j) {
          int64_t p = fill[nd[j]]++;
          c->inv_elem[p] = B.felem - 1 + i;
          c->inv_ln[p] = j;
        }
      }
    }
  }
  for (int n = 0; n < c->nonode; ++n)
    if (c->inv_ptr[n + 1] == c->inv_ptr[n])
      return fail(W3D_ERR_ARG, "w3d_create: node " + std::to_string(n + 1) +
                                   " has no elements");

  // mm10 crystal records of every element of the mm10 blocks
  std::vector<CrystalDev> crys(ncr);
  {
    const int stride = m->angle_stride > 0 ? m->angle_stride : 1;
    for (int b = 0; b < c->nelblk; ++b) {
      const BlockDesc& B = c->blocks[b];
      if (B.model != W3D_MM10) continue;
      c->has_mm10 = true;
      for (int i = 0; i < B.span; ++i)
        for (int k = 0; k < B.ncry; ++k) {
          const double* a =
              m->angles + 3 * ((int64_t)stride * (B.felem - 1 + i) + k);
          if (!mm10_crystal_setup(m->mats[B.mat], a,
                                  &crys[B.crys_off + (int64_t)i * B.ncry + k]))
            return fail(W3D_ERR_UNSUPPORTED, "w3d_create: mm10 crystal");
        }
    }
  }

  // ---- device ----
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  if (hipHostMalloc((void**)&c->h_poll_sc, pin_words(c) * sizeof(double),
                    hipHostMallocPortable | hipHostMallocCoherent) !=
      hipSuccess) {
    c->h_poll_sc = nullptr;
    return fail(W3D_ERR_NOMEM, "w3d_create: pinned memory");
  }
  c->h_rec = c->h_poll_sc + 8;
  for (int k = 0; k < 2; ++k) {
    c->h_poll[k] = reinterpret_cast<int32_t*>(c->h_poll_sc + 4 + k);
    HIPCHK(hipEventCreateWithFlags(&c->poll_ev[k], hipEventDisableTiming));
  }
  int rc;
  if ((rc = upload(&c->d_blocks, c->blocks))) return rc;
  if (!c->trn_idx.empty()) {
    if ((rc = upload(&c->d_trn_idx, c->trn_idx))) return rc;
    if ((rc = upload(&c->d_trn_mat, c->trn_mat))) return rc;
  }
  if ((rc = upload(&c->d_mats, c->mats))) return rc;
  if ((rc = upload(&c->d_therm, c->therm))) return rc;
  if ((rc = upload(&c->d_tables, c->tables))) return rc;
  if ((rc = upload(&c->d_conn, c->conn))) return rc;
  if (c->has_mm10) {
    if ((rc = upload(&c->d_crys, crys))) return rc;
    if ((rc = dalloc(&c->d_uddt, 6 * q))) return rc;
    bool mm10_geonl = false;
    for (const BlockDesc& B : c->blocks)
      mm10_geonl = mm10_geonl || (B.model == W3D_MM10 && B.geonl);
    if (mm10_geonl) {
      if ((rc = dalloc(&c->d_rot_tmp, 9 * q))) return rc;
      if ((rc = dalloc(&c->d_jac_tmp, 9 * (int64_t)c->noelem))) return rc;
    }
    // one work item per 64 consecutive points of an mm10 block
    std::vector<WorkItem> mw;
    for (int b = 0; b < c->nelblk; ++b) {
      const BlockDesc& B = c->blocks[b];
      if (B.model != W3D_MM10) continue;
      const int np = B.span * B.ngp;
      for (int f = 0; f < np; f += 64) {
        WorkItem w;
        w.blk = b;
        w.first = f;
        w.count = std::min(64, np - f);
        w.pad_ = 0;
        mw.push_back(w);
      }
    }
    c->n_work_mm10 = (int)mw.size();
    if ((rc = upload(&c->d_work_mm10, mw))) return rc;
    std::vector<int32_t> mb;
    for (int b = 0; b < c->nelblk; ++b)
      if (c->blocks[b].model == W3D_MM10) mb.push_back(b);
    c->n_mm10_blks = (int)mb.size();
    if ((rc = upload(&c->d_mm10_blks, mb))) return rc;
  }
  {
    std::vector<double> xyz(m->c, m->c + 3 * (int64_t)m->nonode);
    if ((rc = upload(&c->d_coords, xyz))) return rc;
  }
  // (the Ke arrays two words longer: the assembly loads three words of
  // every contribution)
  struct A {
    double** p;
    int64_t n;
  } arrs[] = {{&c->d_stress_n, 9 * q},  {&c->d_stress_n1, 9 * q},
              {&c->d_strain_n, 6 * q},  {&c->d_strain_n1, 6 * q},
              {&c->d_hist_n, h},        {&c->d_hist_n1, h},
              {&c->d_cep, 21 * q},      {&c->d_ek64, ek + 2},
              {&c->d_einfvec, fv},      {&c->d_evol, c->noelem},
              {&c->d_u, 3 * (int64_t)c->nonode},
              {&c->d_du, 3 * (int64_t)c->nonode},
              {&c->d_ifv, 3 * (int64_t)c->nonode},
              {&c->d_blk_sums, kBlkSums * (int64_t)c->nelblk}};
  for (auto& a : arrs) {
    if ((rc = dalloc(a.p, a.n))) return rc;
    HIPCHK(hipMemset(*a.p, 0, std::max<int64_t>(a.n, 1) * sizeof(double)));
  }
  if (c->has_geonl) {  // rotation_init (reopen.f:1840): unit matrices
    std::vector<double> rot(9 * (size_t)q, 0.0);
    for (const BlockDesc& B : c->blocks) {
      const int64_t SG = (int64_t)B.span * B.ngp;
      for (int64_t p = 0; p < SG; ++p)
        for (int k : {0, 4, 8}) rot[9 * B.q_off + k * SG + p] = 1.0;
    }
    if ((rc = upload(&c->d_rot_n, rot))) return rc;
    if ((rc = upload(&c->d_rot_n1, rot))) return rc;
    if ((rc = dalloc(&c->d_u_t, 3 * (int64_t)c->nonode))) return rc;
    if ((rc = dalloc(&c->d_du_t, 3 * (int64_t)c->nonode))) return rc;
    HIPCHK(hipMemset(c->d_u_t, 0, 3 * (size_t)c->nonode * sizeof(double)));
    HIPCHK(hipMemset(c->d_du_t, 0, 3 * (size_t)c->nonode * sizeof(double)));
  }
  if ((rc = dalloc(&c->d_ek32, ek + 2))) return rc;
  HIPCHK(hipMemset(c->d_ek32, 0, (ek + 2) * sizeof(float)));
  if ((rc = dalloc(&c->d_flags, 4))) return rc;
  HIPCHK(hipMemset(c->d_flags, 0, 4 * sizeof(int32_t)));
  if ((rc = dalloc(&c->d_counter, 4))) return rc;
  HIPCHK(hipMemset(c->d_counter, 0, 4 * sizeof(int32_t)));
  HIPCHK(hipDeviceGetAttribute(&c->n_cu, hipDeviceAttributeMultiprocessorCount,
                               c->device));
  // persistent mm10: two waves per SIMD fit (registers), eight per CU
  c->mm10_grid = 8 * std::max(c->n_cu, 1);
  {
    std::vector<WorkItem> items;
    build_work(c, false, items, c->rec_groups, c->rec_start, c->rec_count);
    if ((rc = upload(&c->d_work_rec, items))) return rc;
    // chunk energy partials, and each block's run of chunks (a block's
    // chunks are consecutive in the work list, in element order)
    if ((rc = dalloc(&c->d_en_wg, kBlkSums * items.size()))) return rc;
    std::vector<int32_t> wf(c->nelblk, -1), wc(c->nelblk, 0);
    for (size_t k = 0; k < items.size(); ++k) {
      int b = items[k].blk;
      if (wf[b] < 0) wf[b] = (int32_t)k;
      wc[b] += 1;
    }
    if ((rc = upload(&c->d_blk_wfirst, wf))) return rc;
    if ((rc = upload(&c->d_blk_wcount, wc))) return rc;
    build_work(c, true, items, c->tan_groups, c->tan_start, c->tan_count);
    if ((rc = upload(&c->d_work_tan, items))) return rc;
  }
  if ((rc = dalloc(&c->d_blk_flags, 4 * (int64_t)c->nelblk))) return rc;
  HIPCHK(hipMemset(c->d_blk_flags, 0, 16 * (size_t)c->nelblk));
  if ((rc = dalloc(&c->d_blk_counter, c->nelblk))) return rc;
  HIPCHK(hipMemset(c->d_blk_counter, 0, 4 * (size_t)c->nelblk));
  build_runs(c);
  {
    std::vector<int64_t> off(c->inv_elem.size());
    for (size_t p = 0; p < off.size(); ++p) {
      int e = c->inv_elem[p];
      const BlockDesc& B = c->blocks[c->elem_blk[e]];
      int i = e - (B.felem - 1);
      off[p] = B.ifv_off + (int64_t)i * B.totdof + 3 * c->inv_ln[p];
    }
    if ((rc = upload(&c->d_inv_ptr, c->inv_ptr))) return rc;
    if ((rc = upload(&c->d_inv_off, off))) return rc;
  }
  return W3D_OK;
}

void prof_begin(w3d_ctx* c, int ph) {
  if (!c->profiling || c->capturing || c->nseg[ph] >= 2) return;
  hipEventRecord(c->ev_a[ph][c->nseg[ph]], c->stream);
}
void prof_end(w3d_ctx* c, int ph) {
  if (!c->profiling || c->capturing || c->nseg[ph] >= 2) return;
  hipEventRecord(c->ev_b[ph][c->nseg[ph]], c->stream);
  c->nseg[ph] += 1;
}
// called after the stream has been synchronised: one phase call, the sum
// of its segments
void prof_collect(w3d_ctx* c) {
  if (!c->profiling) return;
  for (int ph = 0; ph < W3D_NUM_PHASES; ++ph) {
    if (!c->nseg[ph]) continue;
    double tot = 0.0;
    bool ok = true;
    for (int k = 0; k < c->nseg[ph]; ++k) {
      float ms = 0.0f;
      ok = ok && hipEventElapsedTime(&ms, c->ev_a[ph][k], c->ev_b[ph][k]) ==
                     hipSuccess;
      tot += ms;
    }
    if (ok) {
      c->prof_ms[ph] += tot;
      c->prof_n[ph] += 1;
    }
    c->nseg[ph] = 0;
  }
}

// A stream for one per-block call: an idle one of the pool, or a new one
// (default priority, non-blocking).
int borrow_stream(w3d_ctx* c, hipStream_t* s) {
  {
    std::lock_guard<std::mutex> lk(c->pool_mu);
    if (!c->pool_idle.empty()) {
      *s = c->pool_idle.back();
      c->pool_idle.pop_back();
      return W3D_OK;
    }
  }
  hipStream_t st;
  HIPCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  std::lock_guard<std::mutex> lk(c->pool_mu);
  c->pool_all.push_back(st);
  *s = st;
  return W3D_OK;
}

void return_stream(w3d_ctx* c, hipStream_t s) {
  std::lock_guard<std::mutex> lk(c->pool_mu);
  c->pool_idle.push_back(s);
}

// The recovery of block b (0-based) on stream s, with the displacements of
// w3d_set_displacements: the block's flags cleared, the first pass, for
// mm10 the material update over the block's own items (its own counter; a
// workgroup for each part of an item: 128 bricks 279 -> 130 us a call),
// grad Fe and the second pass, then the block's sums.
int enqueue_block_recover(w3d_ctx* c, int b, hipStream_t s, int step,
                          int iter, int extrapolated) {
  const w3d_ctx::BlockRuns& R = c->runs[b];
  const int nonlinear = (iter >= 1 || extrapolated) ? 1 : 0;
  const int want_energy = iter > 0 ? 1 : 0;
  DevModel M = c->dev();
  M.flags = c->d_blk_flags + 4 * b;
  const std::vector<int> g{R.rec_key}, st{R.rec_first}, n{R.rec_n};
  int rc = launch_fill_i32(M.flags, 4, 0, s);
  if (!rc)
    rc = launch_recover(M, c->blocks, c->d_work_rec, g, st, n, step, iter,
                        nonlinear, c->d_u, c->d_du, want_energy, c->d_en_wg,
                        0, s);
  if (!rc && R.mm10_n > 0) {
    rc = launch_mm10(M, c->d_work_mm10 + R.mm10_first, R.mm10_n,
                     c->d_blk_counter + b, c->mm10_grid, step,
                     mm10_iter0_off(step, iter, extrapolated), s);
    if (!rc)
      rc = launch_mm10_grads(M, c->d_mm10_blks + R.mm10_idx, 1, b, b + 1,
                             step, s);
    if (!rc)
      rc = launch_recover(M, c->blocks, c->d_work_rec, g, st, n, step, iter,
                          nonlinear, c->d_u, c->d_du, want_energy,
                          c->d_en_wg, 1, s);
  }
  if (!rc && want_energy)
    rc = launch_recover_end(nullptr, nullptr, nullptr, 0, nullptr, c->d_en_wg,
                            c->d_blk_wfirst + b, c->d_blk_wcount + b, 1,
                            c->d_blk_sums + kBlkSums * b, nullptr, nullptr,
                            s);
  return rc;
}

// The status of recovery flags: [0] fatal (mm01), [1] cut, [3] det F <= 0.
int flags_status(const int32_t* f, int step) {
  if (f[0]) return fail(W3D_ERR_NUMERIC, "mm01: negative plastic multiplier");
  // det F <= 0 (fcomp1): a step reduction when one is possible (rstgp1.f)
  if (f[3] && step == 1)
    return fail(W3D_ERR_NUMERIC, "non-positive deformation Jacobian at step 1");
  if (f[1] || f[3]) return W3D_CUT_STEP;
  return W3D_OK;
}

int recover_lists(w3d_ctx* c, RecoverLists& L) {
  L.d_w = c->d_work_rec;
  L.d_wm = c->d_work_mm10;
  L.nwm = c->n_work_mm10;
  L.sg = c->rec_groups;
  L.ss = c->rec_start;
  L.sn = c->rec_count;
  return W3D_OK;
}

int enqueue_recover_stage(w3d_ctx* c, const RecoverLists& L, int stage,
                          int step, int iter, int extrapolated,
                          const double* d_u, const double* d_du, double* d_ifv,
                          bool sums, int first_blk, int nblk) {
  const int nonlinear = (iter >= 1 || extrapolated) ? 1 : 0;
  const int want_energy = (iter > 0) ? 1 : 0;
  DevModel M = c->dev();
  int rc = W3D_OK;
  if (stage == 0) {
    if (c->has_geonl) {
      // the finite-strain update needs u; the tangent later uses X + u + du
      if (!d_u)
        return fail(W3D_ERR_ARG,
                    "recover: finite strains need the displacements u");
    }
    rc = launch_recover_begin(c->d_flags,
                              c->has_geonl ? 3 * (int64_t)c->nonode : 0, d_u,
                              d_du, c->d_u_t, c->d_du_t, c->stream);
    if (rc) return fail(rc, "recover: flag reset launch failed");
    c->last_step = step;
    prof_begin(c, W3D_PHASE_RECOVER);
    rc = launch_recover(M, c->blocks, L.d_w, L.sg, L.ss, L.sn, step, iter,
                        nonlinear, d_u, d_du, want_energy, c->d_en_wg, 0,
                        c->stream);
    prof_end(c, W3D_PHASE_RECOVER);
  } else if (stage == 1) {
    if (L.nwm <= 0) return W3D_OK;
    prof_begin(c, W3D_PHASE_MM10);
    rc = launch_mm10(M, L.d_wm, L.nwm, c->d_counter, c->mm10_grid, step,
                     mm10_iter0_off(step, iter, extrapolated), c->stream);
    prof_end(c, W3D_PHASE_MM10);
  } else if (stage == 2) {
    if (L.nwm <= 0) return W3D_OK;
    prof_begin(c, W3D_PHASE_MM10);
    rc = launch_mm10_grads(M, c->d_mm10_blks, c->n_mm10_blks, first_blk - 1,
                           first_blk - 1 + nblk, step, c->stream);
    prof_end(c, W3D_PHASE_MM10);
  } else {
    if (L.nwm > 0) {
      prof_begin(c, W3D_PHASE_RECOVER);
      rc = launch_recover(M, c->blocks, L.d_w, L.sg, L.ss, L.sn, step, iter,
                          nonlinear, d_u, d_du, want_energy, c->d_en_wg, 1,
                          c->stream);
      prof_end(c, W3D_PHASE_RECOVER);
    }
    // the forces, the energy sums and the host's image in one launch (while
    // phases are timed the forces in a launch of their own)
    const int nsum = sums && want_energy ? c->nelblk : 0;
    const bool apart = c->profiling && !c->capturing && (nsum || L.host);
    if (!rc && d_ifv) {
      prof_begin(c, W3D_PHASE_IFV);
      rc = launch_recover_end(c->d_einfvec, c->d_inv_ptr, c->d_inv_off,
                              c->nonode, d_ifv, c->d_en_wg, c->d_blk_wfirst,
                              c->d_blk_wcount, apart ? 0 : nsum,
                              c->d_blk_sums, c->d_flags,
                              apart ? nullptr : L.host, c->stream);
      prof_end(c, W3D_PHASE_IFV);
      if (rc) return fail(rc, "recover: ifv gather launch failed");
    }
    if (!rc && (nsum || L.host) && (apart || !d_ifv)) {
      prof_begin(c, W3D_PHASE_ENERGY);
      rc = launch_recover_end(nullptr, nullptr, nullptr, 0, nullptr,
                              c->d_en_wg, c->d_blk_wfirst, c->d_blk_wcount,
                              nsum, c->d_blk_sums, c->d_flags, L.host,
                              c->stream);
      prof_end(c, W3D_PHASE_ENERGY);
      if (rc) return fail(rc, "recover: energy reduction launch failed");
    }
  }
  if (rc) return fail(rc, "recover: kernel launch failed");
  return W3D_OK;
}

int enqueue_recover(w3d_ctx* c, const RecoverLists& L, int step, int iter,
                    int extrapolated, const double* d_u, const double* d_du,
                    double* d_ifv, bool sums, int first_blk, int nblk) {
  for (int stage = 0; stage < 4; ++stage) {
    int rc = enqueue_recover_stage(c, L, stage, step, iter, extrapolated, d_u,
                                   d_du, d_ifv, sums, first_blk, nblk);
    if (rc) return rc;
  }
  return W3D_OK;
}

int enqueue_commit(w3d_ctx* c) {
  HIPCHK(hipMemcpyAsync(c->d_stress_n, c->d_stress_n1, 9 * c->nq * 8,
                        hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(c->d_strain_n, c->d_strain_n1, 6 * c->nq * 8,
                        hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(c->d_hist_n, c->d_hist_n1, c->nhist * 8,
                        hipMemcpyDeviceToDevice, c->stream));
  if (c->has_geonl)  // adaptive_saves (mnralg.f:1305)
    HIPCHK(hipMemcpyAsync(c->d_rot_n, c->d_rot_n1, 9 * c->nq * 8,
                          hipMemcpyDeviceToDevice, c->stream));
  return W3D_OK;
}

int enqueue_rollback(w3d_ctx* c) {
  HIPCHK(hipMemcpyAsync(c->d_stress_n1, c->d_stress_n, 9 * c->nq * 8,
                        hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(c->d_strain_n1, c->d_strain_n, 6 * c->nq * 8,
                        hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(c->d_hist_n1, c->d_hist_n, c->nhist * 8,
                        hipMemcpyDeviceToDevice, c->stream));
  if (c->has_geonl)  // adaptive restart (mnralg.f:1393)
    HIPCHK(hipMemcpyAsync(c->d_rot_n1, c->d_rot_n, 9 * c->nq * 8,
                          hipMemcpyDeviceToDevice, c->stream));
  return W3D_OK;
}

int enqueue_csr_values(w3d_ctx* c, const double* d_diag,
                       const double* d_coef) {
  int rc = solver_csr_values(d_diag, d_coef, c->neqns, c->d_csr_vidx,
                             c->csr_nnz, c->d_csr_val, c->stream);
  return rc ? fail(rc, "csr values: launch failed") : W3D_OK;
}

// After the stream: energy and plastic work from the per-block sums (block
// order), then the flags, both from the context's pinned image.
int finish_recover(w3d_ctx* c, int step, int iter, double* energy,
                   double* plastic_work) {
  HIPCHK(hipStreamSynchronize(c->stream));
  double en = 0.0, pw = 0.0, fa = 0.0;
  int nsum = 0;
  if ((energy || plastic_work) && iter > 0) {
    nsum = c->nelblk;
    const double* sums = c->h_rec;
    for (int b = 0; b < nsum; ++b) {
      en = en + sums[kBlkSums * b];
      pw = pw + sums[kBlkSums * b + 1];
      fa = fa + sums[kBlkSums * b + 2];
    }
    c->sum_ifv = fa;
    c->num_term_ifv = c->nifv;
  }
  if (energy) *energy = en;
  if (plastic_work) *plastic_work = pw;
  prof_collect(c);
  int32_t f[4];
  std::memcpy(f, c->h_rec + kBlkSums * nsum, sizeof f);
  return flags_status(f, step);
}

int recover_impl(w3d_ctx* c, int step, int iter, int extrapolated,
                 const double* d_u, const double* d_du, double* d_ifv,
                 double* energy, double* plastic_work, int first_blk,
                 int nblk) {
  HIPCHK(hipSetDevice(c->device));
  RecoverLists L;
  int rc = recover_lists(c, L);
  L.host = c->h_rec;
  if (!rc)
    rc = enqueue_recover(c, L, step, iter, extrapolated, d_u, d_du, d_ifv,
                         energy || plastic_work, first_blk, nblk);
  if (rc) return rc;
  return finish_recover(c, step, iter, energy, plastic_work);
}

// Jacobi-PCG on an assembled matrix (diag, coef device arrays); b and x
// device arrays of neqns (x: initial guess in, solution out).  work: kPcgVectors
// neqns doubles of vectors, tail: kPcgTail.
int pcg_impl(w3d_ctx* c, const double* d_diag, const double* d_coef,
             const double* d_b, double* d_x, double rtol, int maxit,
             int32_t* iters, double* relres, double* work, double* tail) {
  const int n = c->neqns;
  hipStream_t s = c->stream;
  PcgSys S{};
  S.A = c->groups();
  S.val = c->d_csr_val;
  S.diag = d_diag;
  S.b = d_b;
  S.x = d_x;
  S.part = tail + 8;
  S.rtol = rtol;
  S.maxit = maxit;
  S.n = n;
  S.set_work(work);
  S.nwg = pcg_mul_wgs(S.A.ngrp);
  S.single = 1;
  double* sc = tail;
  int32_t* state = reinterpret_cast<int32_t*>(tail + 2);
  int rc = solver_csr_values(d_diag, d_coef, n, c->d_csr_vidx, c->csr_nnz,
                             c->d_csr_val, s);
  // A x, then r = b - A x by the initialisation
  if (!rc) rc = solver_spmv(c->groups(), c->d_csr_val, d_x, S.ax(), s);
  if (!rc) rc = launch_pcg_init(S, s, state, sc);
  const int32_t* st = nullptr;
  if (!rc)
    rc = solve_poll([&](int it) { return launch_pcg_iter(S, it, state, sc, s); },
                    1, maxit, 1, kPollChunk, state, c->h_poll, c->poll_ev, s,
                    &st);
  double v[2] = {0.0, 0.0};  // |b|, r.r
  if (!rc && (hipMemcpyAsync(c->h_poll_sc, sc, sizeof v,
                             hipMemcpyDeviceToHost, s) != hipSuccess ||
              hipStreamSynchronize(s) != hipSuccess))
    rc = W3D_ERR_DEVICE;
  if (rc) return fail(rc, "w3d_solve_pcg: device failure");
  if (st[0] == kPcgZeroRhs) {
    HIPCHK(hipMemsetAsync(d_x, 0, n * sizeof(double), s));
    HIPCHK(hipStreamSynchronize(s));
    if (iters) *iters = 0;
    if (relres) *relres = 0.0;
    return W3D_OK;
  }
  const double rel = std::sqrt(c->h_poll_sc[1]) / c->h_poll_sc[0];
  if (iters) *iters = st[1];
  if (relres) *relres = rel;
  if (st[0] != 1)
    return fail(W3D_ERR_NUMERIC,
                "w3d_solve_pcg: no convergence in " + std::to_string(st[1]) +
                    " iterations (relative residual " +
                    std::to_string(rel) + ")");
  return W3D_OK;
}

// state views ----------------------------------------------------------
struct View {
  double* d = nullptr;
  float* f = nullptr;
  int64_t n = 0;
};

}  // namespace w3d

extern "C" {

const char* w3d_last_error(void) { return g_err.c_str(); }

const char* w3d_version(void) { return "libw3dblk 0.1 (gfx950)"; }

int w3d_create(w3d_ctx** ctx, const w3d_model* model, int device) {
  if (!ctx || !model) return fail(W3D_ERR_ARG, "w3d_create: null argument");
  *ctx = nullptr;
  if (model->abi_version != W3D_ABI_VERSION)
    return fail(W3D_ERR_ARG, "w3d_create: ABI version mismatch");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return fail(W3D_ERR_DEVICE, "w3d_create: no HIP device");
  if (device < 0 || device >= ndev)
    return fail(W3D_ERR_ARG, "w3d_create: bad device ordinal");
  w3d_ctx* c = new w3d_ctx();
  c->device = device;
  const int64_t bytes0 = t_dalloc_bytes;
  int rc = create_impl(c, model);
  c->dev_bytes = t_dalloc_bytes - bytes0;
  if (rc) {
    std::string keep = g_err;
    free_ctx(c);
    delete c;
    g_err = keep;
    return rc;
  }
  *ctx = c;
  return W3D_OK;
}

int w3d_destroy(w3d_ctx* ctx) {
  if (!ctx) return W3D_OK;
  hipSetDevice(ctx->device);
  if (ctx->stream) hipStreamSynchronize(ctx->stream);
  free_ctx(ctx);
  delete ctx;
  return W3D_OK;
}

int w3d_get_blocking(const w3d_ctx* c, int32_t* nelblk, int32_t* elblks) {
  if (!c) return fail(W3D_ERR_ARG, "null context");
  if (nelblk) *nelblk = c->nelblk;
  if (elblks) std::memcpy(elblks, c->elblks.data(), 16 * (size_t)c->nelblk);
  return W3D_OK;
}

int w3d_block_info(const w3d_ctx* c, int32_t blk, int32_t* info5) {
  if (!c || !info5 || blk < 1 || blk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_block_info: bad block");
  const BlockDesc& B = c->blocks[blk - 1];
  info5[0] = B.span;
  info5[1] = B.ngp;
  info5[2] = B.hist;
  info5[3] = B.totdof;
  info5[4] = B.utsz;
  return W3D_OK;
}

int w3d_recover_dev(w3d_ctx* c, int32_t step, int32_t iter,
                    int32_t extrapolated, const double* d_u,
                    const double* d_du, double* d_ifv, double* energy,
                    double* plastic_work) {
  if (!c || !d_du) return fail(W3D_ERR_ARG, "w3d_recover_dev: null argument");
  if (step < 1 || iter < 0) return fail(W3D_ERR_ARG, "w3d_recover: step/iter");
  return recover_impl(c, step, iter, extrapolated, d_u, d_du, d_ifv, energy,
                      plastic_work, 1, c->nelblk);
}

int w3d_recover(w3d_ctx* c, int32_t step, int32_t iter, int32_t extrapolated,
                const double* u, const double* du, double* ifv,
                double* energy, double* plastic_work) {
  if (!c || !du) return fail(W3D_ERR_ARG, "w3d_recover: null argument");
  if (step < 1 || iter < 0) return fail(W3D_ERR_ARG, "w3d_recover: step/iter");
  size_t nb = 3 * (size_t)c->nonode * sizeof(double);
  HIPCHK(hipSetDevice(c->device));
  if (u)
    HIPCHK(hipMemcpyAsync(c->d_u, u, nb, hipMemcpyHostToDevice, c->stream));
  HIPCHK(hipMemcpyAsync(c->d_du, du, nb, hipMemcpyHostToDevice, c->stream));
  int rc = recover_impl(c, step, iter, extrapolated, u ? c->d_u : nullptr,
                        c->d_du, ifv ? c->d_ifv : nullptr, energy,
                        plastic_work, 1, c->nelblk);
  if (rc < 0) return rc;
  if (ifv) {
    HIPCHK(hipMemcpyAsync(ifv, c->d_ifv, nb, hipMemcpyDeviceToHost,
                          c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
  }
  return rc;
}

int w3d_set_displacements(w3d_ctx* c, const double* u, const double* du) {
  if (!c || !du)
    return fail(W3D_ERR_ARG, "w3d_set_displacements: null argument");
  const size_t nb = 3 * (size_t)c->nonode * sizeof(double);
  HIPCHK(hipSetDevice(c->device));
  // earlier work of the context (a commit or rollback) ends first: the
  // per-block calls run on other streams
  HIPCHK(hipStreamSynchronize(c->stream));
  if (u)
    HIPCHK(hipMemcpy(c->d_u, u, nb, hipMemcpyHostToDevice));
  else
    HIPCHK(hipMemset(c->d_u, 0, nb));
  HIPCHK(hipMemcpy(c->d_du, du, nb, hipMemcpyHostToDevice));
  if (c->has_geonl) {  // the tangent's configuration X + u + du
    HIPCHK(hipMemcpy(c->d_u_t, c->d_u, nb, hipMemcpyDeviceToDevice));
    HIPCHK(hipMemcpy(c->d_du_t, c->d_du, nb, hipMemcpyDeviceToDevice));
  }
  c->disp_set = true;
  return W3D_OK;
}

int w3d_recover_block(w3d_ctx* c, int32_t blk, int32_t step, int32_t iter,
                      int32_t extrapolated, double* block_energy,
                      double* block_plastic_work, int32_t* cut) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_recover_block: null context");
  if (blk < 1 || blk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_recover_block: block number");
  if (step < 1 || iter < 0)
    return fail(W3D_ERR_ARG, "w3d_recover_block: step/iter");
  if (!c->disp_set)
    return fail(W3D_ERR_ARG,
                "w3d_recover_block: no w3d_set_displacements before");
  HIPCHK(hipSetDevice(c->device));
  hipStream_t s;
  int rc = borrow_stream(c, &s);
  if (rc) return rc;
  rc = enqueue_block_recover(c, blk - 1, s, step, iter, extrapolated);
  int32_t f[4] = {0, 0, 0, 0};
  double sums[kBlkSums] = {0.0, 0.0, 0.0};
  if (!rc &&
      (hipMemcpyAsync(f, c->d_blk_flags + 4 * (blk - 1), sizeof f,
                      hipMemcpyDeviceToHost, s) != hipSuccess ||
       (iter > 0 &&
        hipMemcpyAsync(sums, c->d_blk_sums + kBlkSums * (blk - 1),
                       sizeof sums, hipMemcpyDeviceToHost, s) != hipSuccess)))
    rc = W3D_ERR_DEVICE;
  if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = W3D_ERR_DEVICE;
  return_stream(c, s);
  if (rc) return fail(rc, "w3d_recover_block: kernel launch failed");
  if (block_energy) *block_energy = sums[0];
  if (block_plastic_work) *block_plastic_work = sums[1];
  rc = flags_status(f, step);
  if (cut) *cut = rc == W3D_CUT_STEP ? 1 : 0;
  return rc;
}

int w3d_recover_blocks(w3d_ctx* c, int32_t first_blk, int32_t nblk,
                       int32_t step, int32_t iter, int32_t extrapolated,
                       const double* u, const double* du) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_recover_blocks: null context");
  if (first_blk < 1 || nblk < 1 || first_blk - 1 + nblk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_recover_blocks: block range");
  if (step < 1 || iter < 0)
    return fail(W3D_ERR_ARG, "w3d_recover_blocks: step/iter");
  int rc;
  if (du && (rc = w3d_set_displacements(c, u, du))) return rc;
  if (!c->disp_set)
    return fail(W3D_ERR_ARG, "w3d_recover_blocks: no displacements");
  HIPCHK(hipSetDevice(c->device));
  hipStream_t s;
  if ((rc = borrow_stream(c, &s))) return rc;
  for (int b = first_blk - 1; b < first_blk - 1 + nblk && !rc; ++b)
    rc = enqueue_block_recover(c, b, s, step, iter, extrapolated);
  std::vector<int32_t> f(4 * (size_t)nblk, 0);
  if (!rc && hipMemcpyAsync(f.data(), c->d_blk_flags + 4 * (first_blk - 1),
                            f.size() * 4, hipMemcpyDeviceToHost,
                            s) != hipSuccess)
    rc = W3D_ERR_DEVICE;
  if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = W3D_ERR_DEVICE;
  return_stream(c, s);
  if (rc) return fail(rc, "w3d_recover_blocks: kernel launch failed");
  int32_t any[4] = {0, 0, 0, 0};
  for (int b = 0; b < nblk; ++b)
    for (int k = 0; k < 4; ++k) any[k] |= f[4 * b + k];
  return flags_status(any, step);
}

int w3d_assemble_ifv(w3d_ctx* c, double* ifv, double* sum_ifv,
                     int64_t* num_term_ifv) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_assemble_ifv: null context");
  HIPCHK(hipSetDevice(c->device));
  int rc = launch_recover_end(c->d_einfvec, c->d_inv_ptr, c->d_inv_off,
                              c->nonode, c->d_ifv, nullptr, nullptr, nullptr,
                              0, nullptr, nullptr, nullptr, c->stream);
  if (rc) return fail(rc, "w3d_assemble_ifv: launch failed");
  if (ifv)
    HIPCHK(hipMemcpyAsync(ifv, c->d_ifv, 3 * (size_t)c->nonode * 8,
                          hipMemcpyDeviceToHost, c->stream));
  std::vector<double> sums;
  if (sum_ifv) {  // the blocks' sums of the last per-block recoveries
    sums.resize(kBlkSums * (size_t)c->nelblk);
    HIPCHK(hipMemcpyAsync(sums.data(), c->d_blk_sums, sums.size() * 8,
                          hipMemcpyDeviceToHost, c->stream));
  }
  HIPCHK(hipStreamSynchronize(c->stream));
  if (sum_ifv) {
    double fa = 0.0;
    for (int b = 0; b < c->nelblk; ++b) fa = fa + sums[kBlkSums * b + 2];
    *sum_ifv = fa;
  }
  if (num_term_ifv) *num_term_ifv = c->nifv;
  return W3D_OK;
}

int w3d_get_ifv_sums(const w3d_ctx* c, double* sum_ifv,
                     int64_t* num_term_ifv) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_get_ifv_sums: null context");
  if (sum_ifv) *sum_ifv = c->sum_ifv;
  if (num_term_ifv) *num_term_ifv = c->num_term_ifv;
  return W3D_OK;
}

// bdbt_asym for every element (asymmetric assembly), FP64
static int tangent_full(w3d_ctx* c) {
  int rc;
  prof_begin(c, W3D_PHASE_TANGENT);
  rc = launch_tangent_full(c->dev(), c->d_work_tan, c->tan_groups,
                           c->tan_start, c->tan_count, c->d_ekf_off, c->d_ekf,
                           c->stream);
  prof_end(c, W3D_PHASE_TANGENT);
  if (rc) return fail(rc, "w3d_tangent: full Ke launch failed");
  c->tangent_precision = W3D_FP64;
  c->asym_tangent = true;
  c->csr_asym_ready = false;
  HIPCHK(hipStreamSynchronize(c->stream));
  prof_collect(c);
  return W3D_OK;
}

// The tangents of blocks [first, first + nblk) (0-based) on stream s.
static int enqueue_block_tangents(w3d_ctx* c, int first, int nblk,
                                  int precision, hipStream_t s) {
  DevModel M = c->dev();
  int rc = W3D_OK;
  for (int b = first; b < first + nblk && !rc; ++b) {
    const w3d_ctx::BlockRuns& R = c->runs[b];
    const std::vector<int> g{R.tan_key}, st{R.tan_first}, n{R.tan_n};
    if (c->asym)
      rc = launch_tangent_full(M, c->d_work_tan, g, st, n, c->d_ekf_off,
                               c->d_ekf, s);
    else
      rc = launch_tangent_mfma(M, c->d_work_tan, g, st, n, precision, s);
  }
  return rc;
}

static int tangent_args(w3d_ctx* c, int precision, bool whole) {
  if (precision != W3D_FP64 && precision != W3D_FP32)
    return fail(W3D_ERR_ARG, "w3d_tangent: precision");
  if (c->asym && precision != W3D_FP64)
    return fail(W3D_ERR_UNSUPPORTED,
                "w3d_tangent: asymmetric assembly takes the FP64 tangent");
  (void)whole;
  return W3D_OK;
}

int w3d_tangent_block(w3d_ctx* c, int32_t blk, int32_t step, int32_t iter,
                      int32_t precision) {
  (void)step;
  (void)iter;
  if (!c) return fail(W3D_ERR_ARG, "w3d_tangent_block: null context");
  if (blk < 1 || blk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_tangent_block: block number");
  int rc = tangent_args(c, precision, false);
  if (rc) return rc;
  HIPCHK(hipSetDevice(c->device));
  hipStream_t s;
  if ((rc = borrow_stream(c, &s))) return rc;
  {
    // the context records which Ke array the blocks' tangents are in
    std::lock_guard<std::mutex> lk(c->pool_mu);
    c->tangent_precision = precision;
    if (c->asym) {
      c->asym_tangent = true;
      c->csr_asym_ready = false;
    }
  }
  rc = enqueue_block_tangents(c, blk - 1, 1, precision, s);
  if (hipStreamSynchronize(s) != hipSuccess && !rc) rc = W3D_ERR_DEVICE;
  return_stream(c, s);
  if (rc) return fail(rc, "w3d_tangent_block: kernel launch failed");
  return W3D_OK;
}

int w3d_tangent_blocks(w3d_ctx* c, int32_t first_blk, int32_t nblk,
                       int32_t step, int32_t iter, int32_t precision) {
  (void)step;
  (void)iter;
  if (!c) return fail(W3D_ERR_ARG, "w3d_tangent: null context");
  if (first_blk < 1 || nblk < 1 || first_blk - 1 + nblk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_tangent_blocks: block range");
  int rc = tangent_args(c, precision, first_blk == 1 && nblk == c->nelblk);
  if (rc) return rc;
  HIPCHK(hipSetDevice(c->device));
  if (first_blk == 1 && nblk == c->nelblk) {  // one launch per group
    if (c->asym) return tangent_full(c);
    prof_begin(c, W3D_PHASE_TANGENT);
    rc = launch_tangent_mfma(c->dev(), c->d_work_tan, c->tan_groups,
                             c->tan_start, c->tan_count, precision,
                             c->stream);
    prof_end(c, W3D_PHASE_TANGENT);
  } else {
    if (c->asym) {
      c->asym_tangent = true;
      c->csr_asym_ready = false;
    }
    rc = enqueue_block_tangents(c, first_blk - 1, nblk, precision, c->stream);
  }
  if (rc) return fail(rc, "w3d_tangent: kernel launch failed");
  c->tangent_precision = precision;
  HIPCHK(hipStreamSynchronize(c->stream));
  prof_collect(c);
  return W3D_OK;
}

int w3d_tangent(w3d_ctx* c, int32_t step, int32_t iter, int32_t precision) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_tangent: null context");
  return w3d_tangent_blocks(c, 1, c->nelblk, step, iter, precision);
}

static int finish_pattern(w3d_ctx* c, int32_t* neqns_out,
                          int64_t* ncoeff_out, int64_t bytes0);

int w3d_pattern(w3d_ctx* c, const int32_t* cstmap, int32_t* neqns_out,
                int64_t* ncoeff_out) {
  if (!c || !cstmap) return fail(W3D_ERR_ARG, "w3d_pattern: null argument");
  const int64_t bytes0 = t_dalloc_bytes;
  const int nd = 3 * c->nonode;
  // dof_map (assemble_code.f:561)
  c->dof_eqn_map.assign(nd, 0);
  c->eqn_node_map.assign(nd, 0);
  int neq = 0;
  for (int d = 1; d <= nd; ++d) {
    if (cstmap[d - 1] != 0) continue;
    neq = neq + 1;
    c->dof_eqn_map[d - 1] = neq;
    c->eqn_node_map[neq - 1] = (d - 1) / 3 + 1;
  }
  c->eqn_node_map.resize(neq);
  c->neqns = neq;
  // rows of the upper triangle (build_col_sparse_symm_srow): columns of the
  // row's node's elements right of the diagonal, sorted, unique
  std::vector<std::vector<int32_t>> rows(neq > 0 ? neq : 1);
  c->k_ptrs.assign(neq, 0);
#pragma omp parallel for schedule(dynamic, 256)
  for (int srow = 1; srow <= neq - 1; ++srow) {
    int snode = c->eqn_node_map[srow - 1] - 1;
    std::vector<int32_t>& list = rows[srow - 1];
    for (int64_t p = c->inv_ptr[snode]; p < c->inv_ptr[snode + 1]; ++p) {
      int e = c->inv_elem[p];
      const BlockDesc& B = c->blocks[c->elem_blk[e]];
      const int32_t* nd_ = &c->conn[B.conn_off + (int64_t)(e - (B.felem - 1)) * B.nnode];
      for (int ecol = 0; ecol < B.totdof; ++ecol) {
        int cmp = ecol / B.nnode, j = ecol % B.nnode;
        int scol = c->dof_eqn_map[3 * nd_[j] + cmp];
        if (scol <= srow) continue;
        list.push_back(scol);
      }
    }
    std::sort(list.begin(), list.end());
    list.erase(std::unique(list.begin(), list.end()), list.end());
    c->k_ptrs[srow - 1] = (int32_t)list.size();
  }
  c->row_start.assign(neq + 1, 0);
  for (int r = 0; r < neq; ++r) c->row_start[r + 1] = c->row_start[r] + c->k_ptrs[r];
  c->ncoeff = c->row_start[neq];
  c->k_indexes.resize(c->ncoeff);
  for (int r = 0; r < neq; ++r)
    if (!rows[r].empty())
      std::memcpy(&c->k_indexes[c->row_start[r]], rows[r].data(),
                  rows[r].size() * sizeof(int32_t));
  rows.clear();
  HIPCHK(hipSetDevice(c->device));
  dfree(c->d_asm_hdr);
  dfree(c->d_asm_src);
  dfree(c->d_asm_wbase);
  dfree(c->d_kout);
  c->asm_ready = false;
  // assembly map (assem_by_row / assem_a_row, assemble_code.f:659,785).
  // Outputs: the diagonal of row r at t = r, coefficient k of the upper
  // triangle at t = neqns + k.  They are cut into segments: one per
  // diagonal, then, row by row, one per further component of the row's own
  // node and one per higher column node m covering m's components.  A
  // segment lists one Ke word per contribution, in the reference's order:
  // elements on the row's node in inverse-incidence order, then every local
  // occurrence of the row's node (erow), then of the column node (ecol).
  // Component c' of a column-node segment reads that word + c' (row-major
  // ranked layout: the element's columns of one node are consecutive).
  // Header: contributions | component mask << 8.  Per 64 segments: the
  // index of their first contribution and of their first output.
  struct Occ {
    int m;          // global node (0-based) at a local position
    int k;          // element's place in the row node's element list
    int64_t base;   // first Ke word of the element
    int td;         // element dofs
    int rank;       // rank of the local position
  };
  const int64_t nout = (int64_t)neq + c->ncoeff;
  // occurrences of nodes >= n in the elements on n, sorted by (node,
  // element) with local positions ascending; self = occurrences of n
  auto node_occ = [&](int n, std::vector<Occ>& occ, std::vector<Occ>& self) {
    occ.clear();
    self.clear();
    int k = 0;
    for (int64_t p = c->inv_ptr[n]; p < c->inv_ptr[n + 1]; ++p, ++k) {
      int e = c->inv_elem[p];
      const BlockDesc& B = c->blocks[c->elem_blk[e]];
      int i = e - (B.felem - 1);
      const int32_t* nd_ = &c->conn[B.conn_off + (int64_t)i * B.nnode];
      int rank[kMaxNodes];
      node_ranks(nd_, B.nnode, rank);
      int64_t base = B.ek_off + (int64_t)i * B.utsz;
      for (int b = 0; b < B.nnode; ++b) {
        if (nd_[b] < n) continue;
        Occ o{nd_[b], k, base, B.totdof, rank[b]};
        if (nd_[b] == n) self.push_back(o);
        else occ.push_back(o);
      }
    }
    std::stable_sort(occ.begin(), occ.end(), [](const Occ& x, const Occ& y) {
      return x.m != y.m ? x.m < y.m : x.k < y.k;
    });
  };
  auto word = [](const Occ& a, int ca, const Occ& b, int cb) -> int64_t {
    int p = 3 * a.rank + ca, q = 3 * b.rank + cb;
    return a.base + (p <= q ? ek_word(a.td, p, q) : ek_word(a.td, q, p));
  };
  // contributions of row occurrences `self` against column occurrences
  // col[y0, y1) (sorted by element), element by element
  auto pairs = [](const std::vector<Occ>& self, const std::vector<Occ>& col,
                  size_t y0, size_t y1, auto&& f) {
    for (size_t x = 0; x < self.size();) {
      size_t x1 = x;
      while (x1 < self.size() && self[x1].k == self[x].k) ++x1;
      size_t y = y0;
      while (y < y1 && col[y].k < self[x].k) ++y;
      for (size_t xx = x; xx < x1; ++xx)
        for (size_t yy = y; yy < y1 && col[yy].k == self[x].k; ++yy)
          f(self[xx], col[yy]);
      x = x1;
    }
  };
  // segments of the rows of node n, in output order:
  // seg(row component, coefficient?, kernel mask, column node, column
  // components, body(emit))
  auto walk = [&](int n, const std::vector<Occ>& occ,
                  const std::vector<Occ>& self, auto&& seg) {
    for (int ca = 0; ca < 3; ++ca) {
      if (c->dof_eqn_map[3 * n + ca] == 0) continue;
      seg(ca, false, 1, n, 1 << ca, [&](auto&& emit) {
        pairs(self, self, 0, self.size(),
              [&](const Occ& a, const Occ& b) { emit(word(a, ca, b, ca)); });
      });
      for (int cb = ca + 1; cb < 3; ++cb) {
        if (c->dof_eqn_map[3 * n + cb] == 0) continue;
        seg(ca, true, 1, n, 1 << cb, [&](auto&& emit) {
          pairs(self, self, 0, self.size(),
                [&](const Occ& a, const Occ& b) { emit(word(a, ca, b, cb)); });
        });
      }
      for (size_t g = 0; g < occ.size();) {
        size_t h = g;
        while (h < occ.size() && occ[h].m == occ[g].m) ++h;
        const int m = occ[g].m;
        int mask = 0;
        for (int cb = 0; cb < 3; ++cb)
          if (c->dof_eqn_map[3 * m + cb] != 0) mask |= 1 << cb;
        if (mask)
          seg(ca, true, mask, m, mask, [&](auto&& emit) {
            pairs(self, occ, g, h,
                  [&](const Occ& a, const Occ& b) { emit(word(a, ca, b, 0)); });
          });
        g = h;
      }
    }
  };
  std::vector<int64_t> nseg_row(neq, 0), nsrc_diag(neq, 0), nsrc_coef(neq, 0);
  int bad = 0;
#pragma omp parallel
  {
    std::vector<Occ> occ, self;
#pragma omp for schedule(dynamic, 64) reduction(max : bad)
    for (int n = 0; n < c->nonode; ++n) {
      node_occ(n, occ, self);
      walk(n, occ, self, [&](int ca, bool coef, int, int, int, auto&& body) {
        const int srow = c->dof_eqn_map[3 * n + ca];
        int64_t cnt = 0;
        body([&](int64_t) { ++cnt; });
        if (cnt > 255) bad = 1;
        if (coef) {
          nseg_row[srow - 1] += 1;
          nsrc_coef[srow - 1] += cnt;
        } else {
          nsrc_diag[srow - 1] = cnt;
        }
      });
    }
  }
  if (bad)
    return fail(W3D_ERR_UNSUPPORTED,
                "w3d_pattern: more than 255 contributions to one coefficient");
  std::vector<int64_t> seg_off(neq + 1, 0), src_diag(neq + 1, 0),
      src_coef(neq + 1, 0);
  for (int r = 0; r < neq; ++r) {
    seg_off[r + 1] = seg_off[r] + nseg_row[r];
    src_diag[r + 1] = src_diag[r] + nsrc_diag[r];
    src_coef[r + 1] = src_coef[r] + nsrc_coef[r];
  }
  const int64_t nseg = neq + seg_off[neq];
  const int64_t nsrc = src_diag[neq] + src_coef[neq];
  std::vector<uint16_t> hdr(nseg);
  std::vector<uint32_t> src(nsrc);
#pragma omp parallel
  {
    std::vector<Occ> occ, self;
#pragma omp for schedule(dynamic, 64) reduction(max : bad)
    for (int n = 0; n < c->nonode; ++n) {
      node_occ(n, occ, self);
      int64_t sg[3], sc[3], kp[3];
      for (int ca = 0; ca < 3; ++ca) {
        const int srow = c->dof_eqn_map[3 * n + ca];
        if (srow == 0) continue;
        sg[ca] = neq + seg_off[srow - 1];
        sc[ca] = src_diag[neq] + src_coef[srow - 1];
        kp[ca] = 0;
      }
      walk(n, occ, self, [&](int ca, bool coef, int kmask, int m, int cols,
                             auto&& body) {
        const int srow = c->dof_eqn_map[3 * n + ca];
        int64_t pos = coef ? sc[ca] : src_diag[srow - 1];
        const int64_t p0 = pos;
        body([&](int64_t w) { src[pos++] = (uint32_t)w; });
        const int cnt = (int)(pos - p0);
        if (!coef) {
          hdr[srow - 1] = (uint16_t)(cnt | 1 << 8);
          return;
        }
        sc[ca] = pos;
        hdr[sg[ca]++] = (uint16_t)(cnt | kmask << 8);
        // the segment's outputs are the row's next coefficients
        const int32_t* kidx = c->k_indexes.data() + c->row_start[srow - 1];
        for (int cb = 0; cb < 3; ++cb) {
          if (!(cols >> cb & 1)) continue;
          if (kp[ca] >= c->k_ptrs[srow - 1] ||
              kidx[kp[ca]] != c->dof_eqn_map[3 * m + cb])
            bad = 1;
          ++kp[ca];
        }
      });
      for (int ca = 0; ca < 3; ++ca) {
        const int srow = c->dof_eqn_map[3 * n + ca];
        if (srow != 0 && kp[ca] != c->k_ptrs[srow - 1]) bad = 1;
      }
    }
  }
  if (bad)
    return fail(W3D_ERR_NUMERIC, "w3d_pattern: assembly map does not match "
                                 "the sparsity pattern");
  const int64_t nwave = (nseg + 63) / 64;
  std::vector<int64_t> wbase(2 * std::max<int64_t>(nwave, 1), 0);
  {
    int64_t so = 0, oo = 0;
    for (int64_t t = 0; t < nseg; ++t) {
      if (t % 64 == 0) {
        wbase[2 * (t / 64)] = so;
        wbase[2 * (t / 64) + 1] = oo;
      }
      so += hdr[t] & 255;
      oo += __builtin_popcount(hdr[t] >> 8);
    }
    if (oo != nout)
      return fail(W3D_ERR_NUMERIC, "w3d_pattern: assembly map output count");
  }
  c->asm_nseg = nseg;
  int rc;
  if ((rc = upload(&c->d_asm_hdr, hdr))) return rc;
  if ((rc = upload(&c->d_asm_src, src))) return rc;
  if ((rc = upload(&c->d_asm_wbase, wbase))) return rc;
  if ((rc = dalloc(&c->d_kout, nout))) return rc;
  c->asm_ready = true;
  return finish_pattern(c, neqns_out, ncoeff_out, bytes0);
}

// The rest of w3d_pattern once the assembly map is built: the solver's
// full symmetric CSR and the outputs.
static int finish_pattern(w3d_ctx* c, int32_t* neqns_out,
                          int64_t* ncoeff_out, int64_t bytes0) {
  const int neq = c->neqns;
  int rc;
  // full symmetric CSR for the solver: row j = the transposed upper entries
  // (i, j) of rows i < j (ascending i), the diagonal, then row j's upper
  // entries (ascending columns)
  {
    std::vector<int64_t> low(neq + 1, 0);
    for (int64_t k = 0; k < c->ncoeff; ++k) low[c->k_indexes[k] - 1 + 1] += 1;
    std::vector<int64_t> rp(neq + 1, 0);
    for (int r = 0; r < neq; ++r)
      rp[r + 1] = rp[r] + low[r + 1] + 1 + c->k_ptrs[r];
    const int64_t nnz = rp[neq];
    c->csr_maxrow = 0;
    for (int r = 0; r < neq; ++r)
      c->csr_maxrow = std::max<int>(c->csr_maxrow, (int)(rp[r + 1] - rp[r]));
    std::vector<int32_t> col(nnz);
    std::vector<uint32_t> vidx(nnz);
    std::vector<int64_t> fill(neq);
    for (int r = 0; r < neq; ++r) fill[r] = rp[r];
    for (int r = 0; r < neq; ++r) {
      for (int64_t k = c->row_start[r]; k < c->row_start[r + 1]; ++k) {
        int j = c->k_indexes[k] - 1;
        int64_t f = fill[j]++;
        col[f] = r;
        vidx[f] = (uint32_t)(neq + k);
      }
    }
    // rows in groups that share their columns: the consecutive equations
    // of one node (a row's columns compared with the row before it, while
    // they are at hand; a parallel loop here, the last of the set-up, left
    // its threads spinning for 200 ms beside the caller's first iterations)
    std::vector<RowGroup> grp;
    for (int r = 0; r < neq; ++r) {
      int64_t f = fill[r];
      col[f] = r;
      vidx[f] = (uint32_t)r;
      ++f;
      for (int64_t k = c->row_start[r]; k < c->row_start[r + 1]; ++k, ++f) {
        col[f] = c->k_indexes[k] - 1;
        vidx[f] = (uint32_t)(neq + k);
      }
      const int32_t len = (int32_t)(rp[r + 1] - rp[r]);
      if (r > 0 && c->eqn_node_map[r] == c->eqn_node_map[r - 1] &&
          grp.back().len() == len && grp.back().rows() < 3 &&
          std::equal(col.begin() + rp[r], col.begin() + rp[r + 1],
                     col.begin() + rp[r - 1]))
        grp.back().nl += 1;
      else
        grp.push_back({rp[r], r, len << 2 | 1});
    }
    dfree(c->d_csr_rp);
    dfree(c->d_csr_col);
    dfree(c->d_csr_vidx);
    dfree(c->d_csr_val);
    dfree(c->d_pcg);
    dfree(c->d_bicg);
    dfree(c->d_fa_eqdof);
    if ((rc = upload(&c->d_csr_rp, rp))) return rc;
    if ((rc = upload(&c->d_csr_col, col))) return rc;
    if ((rc = upload(&c->d_csr_vidx, vidx))) return rc;
    if ((rc = dalloc(&c->d_csr_val, nnz))) return rc;
    c->csr_ngrp = (int)grp.size();
    dfree(c->d_csr_grp);
    if ((rc = upload(&c->d_csr_grp, grp))) return rc;
    // the solver's work array and its tail, b and x
    if ((rc = dalloc(&c->d_pcg, (kPcgVectors + 2) * (int64_t)neq + kPcgTail)))
      return rc;
    c->csr_nnz = nnz;
    c->csr_serial = -1;
    c->assembled = 0;
  }
  c->dev_bytes += t_dalloc_bytes - bytes0;
  if (neqns_out) *neqns_out = neq;
  if (ncoeff_out) *ncoeff_out = c->ncoeff;
  return W3D_OK;
}

int w3d_get_pattern(const w3d_ctx* c, int32_t* dof_eqn_map,
                    int32_t* eqn_node_map, int32_t* k_ptrs,
                    int32_t* k_indexes) {
  if (!c || c->dof_eqn_map.empty())
    return fail(W3D_ERR_ARG, "w3d_get_pattern: no pattern");
  if (dof_eqn_map)
    std::memcpy(dof_eqn_map, c->dof_eqn_map.data(), 12 * (size_t)c->nonode);
  if (eqn_node_map)
    std::memcpy(eqn_node_map, c->eqn_node_map.data(), 4 * (size_t)c->neqns);
  if (k_ptrs) std::memcpy(k_ptrs, c->k_ptrs.data(), 4 * (size_t)c->neqns);
  if (k_indexes)
    std::memcpy(k_indexes, c->k_indexes.data(), 4 * (size_t)c->ncoeff);
  return W3D_OK;
}

int w3d_set_asymmetric(w3d_ctx* c, int32_t on) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_set_asymmetric: null context");
  if (on)
    for (const BlockDesc& B : c->blocks) {
      if (B.geonl)
        return fail(W3D_ERR_UNSUPPORTED,
                    "w3d_set_asymmetric: finite-strain blocks");
      if (B.trn)
        return fail(W3D_ERR_UNSUPPORTED,
                    "w3d_set_asymmetric: skewed constraints");
    }
  if (on && !c->d_ekf) {  // the full Ke of every element
    std::vector<int64_t> off(c->nelblk + 1, 0);
    for (int b = 0; b < c->nelblk; ++b) {
      const BlockDesc& B = c->blocks[b];
      off[b + 1] = off[b] + (int64_t)B.span * B.totdof * B.totdof;
    }
    c->n_ekf = off[c->nelblk];
    const int64_t bytes0 = t_dalloc_bytes;
    int rc;
    HIPCHK(hipSetDevice(c->device));
    if ((rc = upload(&c->d_ekf_off, off))) return rc;
    if ((rc = dalloc(&c->d_ekf, c->n_ekf))) return rc;
    c->dev_bytes += t_dalloc_bytes - bytes0;
  }
  c->asym = on != 0;
  c->asym_tangent = false;
  c->csr_asym_ready = false;
  c->tangent_precision = -1;
  return W3D_OK;
}

int w3d_get_csr_pattern(const w3d_ctx* c, int64_t* nnz, int64_t* rp,
                        int32_t* col) {
  if (!c || !c->d_csr_rp)
    return fail(W3D_ERR_ARG, "w3d_get_csr_pattern: no pattern");
  HIPCHK(hipSetDevice(c->device));
  if (nnz) *nnz = c->csr_nnz;
  if (rp)
    HIPCHK(hipMemcpy(rp, c->d_csr_rp, 8 * (size_t)(c->neqns + 1),
                     hipMemcpyDeviceToHost));
  if (col && c->csr_nnz)
    HIPCHK(hipMemcpy(col, c->d_csr_col, 4 * (size_t)c->csr_nnz,
                     hipMemcpyDeviceToHost));
  return W3D_OK;
}

int w3d_assemble_csr_dev(w3d_ctx* c, double* d_val) {
  if (!c || !c->d_csr_rp)
    return fail(W3D_ERR_ARG, "w3d_assemble_csr: no pattern");
  if (!c->asym || !c->asym_tangent)
    return fail(W3D_ERR_ARG,
                "w3d_assemble_csr: no full Ke (asymmetric assembly off, or "
                "no tangent since it was switched on)");
  if (!d_val && c->csr_nnz) return fail(W3D_ERR_ARG, "w3d_assemble_csr: null");
  if (c->csr_maxrow > kAsmMaxRow)
    return fail(W3D_ERR_UNSUPPORTED,
                "w3d_assemble_csr: a row couples more than " +
                    std::to_string(kAsmMaxRow) + " equations");
  HIPCHK(hipSetDevice(c->device));
  int rc;
  if (!c->d_fa_eqdof) {
    // the gather map (once per pattern): per (node, element) incidence p,
    // the element's Ke base and, per element column, its position in the
    // node's CSR rows (the three rows of a node share their columns)
    const int64_t bytes0 = t_dalloc_bytes;
    const int neq = c->neqns;
    std::vector<int32_t> eqdof(neq > 0 ? neq : 1, 0);
    for (int d = 0; d < 3 * c->nonode; ++d)
      if (c->dof_eqn_map[d]) eqdof[c->dof_eqn_map[d] - 1] = d;
    std::vector<int64_t> rp(neq + 1);
    std::vector<int32_t> col(c->csr_nnz > 0 ? c->csr_nnz : 1);
    HIPCHK(hipMemcpy(rp.data(), c->d_csr_rp, 8 * (size_t)(neq + 1),
                     hipMemcpyDeviceToHost));
    if (c->csr_nnz)
      HIPCHK(hipMemcpy(col.data(), c->d_csr_col, 4 * (size_t)c->csr_nnz,
                       hipMemcpyDeviceToHost));
    std::vector<int64_t> boff(c->nelblk + 1, 0);
    for (int b = 0; b < c->nelblk; ++b)
      boff[b + 1] = boff[b] + (int64_t)c->blocks[b].span *
                                  c->blocks[b].totdof * c->blocks[b].totdof;
    const int64_t ninv = c->inv_ptr[c->nonode];
    std::vector<int64_t> ebase(ninv > 0 ? ninv : 1), atoff(ninv + 1, 0);
    for (int64_t p = 0; p < ninv; ++p) {
      const BlockDesc& B = c->blocks[c->elem_blk[c->inv_elem[p]]];
      atoff[p + 1] = atoff[p] + B.totdof;
    }
    std::vector<uint16_t> at(atoff[ninv] > 0 ? atoff[ninv] : 1, kAsmNone);
    for (int n = 0; n < c->nonode; ++n) {
      int r = -1;  // a free row of the node
      for (int k = 0; k < 3 && r < 0; ++k)
        if (c->dof_eqn_map[3 * n + k]) r = c->dof_eqn_map[3 * n + k] - 1;
      for (int k = 0; k < 3 && r >= 0; ++k) {  // the rows share columns
        const int q = c->dof_eqn_map[3 * n + k] - 1;
        if (q < 0) continue;
        if (rp[q + 1] - rp[q] != rp[r + 1] - rp[r] ||
            !std::equal(col.begin() + rp[q], col.begin() + rp[q + 1],
                        col.begin() + rp[r]))
          return fail(W3D_ERR_ARG,
                      "w3d_assemble_csr: rows of a node differ in columns");
      }
      for (int64_t p = c->inv_ptr[n]; p < c->inv_ptr[n + 1]; ++p) {
        const int e = c->inv_elem[p], b = c->elem_blk[e];
        const BlockDesc& B = c->blocks[b];
        const int NN = B.nnode, T = B.totdof, i = e - (B.felem - 1);
        ebase[p] = boff[b] + (int64_t)i * T * T;
        if (r < 0) continue;
        const int32_t* cb = col.data() + rp[r];
        const int32_t* ce = col.data() + rp[r + 1];
        for (int ecol = 0; ecol < T; ++ecol) {
          const int nd = c->conn[B.conn_off + (int64_t)i * NN + ecol % NN];
          const int scol = c->dof_eqn_map[3 * nd + ecol / NN];
          if (scol == 0) continue;
          const int32_t* f = std::lower_bound(cb, ce, scol - 1);
          if (f == ce || *f != scol - 1)
            return fail(W3D_ERR_ARG, "w3d_assemble_csr: pattern lacks a column");
          at[atoff[p] + ecol] = (uint16_t)(f - cb);
        }
      }
    }
    dfree(c->d_fa_invptr); dfree(c->d_fa_ln); dfree(c->d_fa_ebase);
    dfree(c->d_fa_atoff); dfree(c->d_fa_at);
    if ((rc = upload(&c->d_fa_eqdof, eqdof))) return rc;
    if ((rc = upload(&c->d_fa_invptr, c->inv_ptr))) return rc;
    if ((rc = upload(&c->d_fa_ln, c->inv_ln))) return rc;
    if ((rc = upload(&c->d_fa_ebase, ebase))) return rc;
    if ((rc = upload(&c->d_fa_atoff, atoff))) return rc;
    if ((rc = upload(&c->d_fa_at, at))) return rc;
    // the BiCGStab vectors of this pattern: b, x and the work array
    dfree(c->d_bicg);
    if ((rc = dalloc(&c->d_bicg, 2 * (int64_t)neq +
                                     bicgstab_words(neq, c->csr_ngrp))))
      return rc;
    c->dev_bytes += t_dalloc_bytes - bytes0;
  }
  prof_begin(c, W3D_PHASE_ASSEMBLE);
  rc = launch_assemble_full(c->d_ekf, c->d_fa_ebase, c->d_fa_atoff,
                            c->d_fa_at, c->d_fa_eqdof, c->d_fa_invptr,
                            c->d_fa_ln, c->groups(), c->csr_maxrow, d_val,
                            c->stream);
  prof_end(c, W3D_PHASE_ASSEMBLE);
  if (rc) return fail(rc, "w3d_assemble_csr: kernel launch failed");
  HIPCHK(hipStreamSynchronize(c->stream));
  prof_collect(c);
  return W3D_OK;
}

int w3d_assemble_csr(w3d_ctx* c, double* val) {
  int rc = w3d_assemble_csr_dev(c, c ? c->d_csr_val : nullptr);
  if (rc) return rc;
  if (val && c->csr_nnz)
    HIPCHK(hipMemcpy(val, c->d_csr_val, 8 * (size_t)c->csr_nnz,
                     hipMemcpyDeviceToHost));
  c->csr_serial = -1;  // the solver's CSR values are no longer the VSS's
  c->csr_asym_ready = true;
  return W3D_OK;
}

int w3d_solve_bicgstab(w3d_ctx* c, const double* rhs, double* x, double rtol,
                       int32_t maxit, int32_t* iters, double* relres) {
  if (!c || !c->d_csr_rp)
    return fail(W3D_ERR_ARG, "w3d_solve_bicgstab: no pattern");
  if (!c->asym || !c->csr_asym_ready)
    return fail(W3D_ERR_ARG, "w3d_solve_bicgstab: no w3d_assemble_csr since "
                             "the last tangent");
  if (!rhs || !x) return fail(W3D_ERR_ARG, "w3d_solve_bicgstab: null argument");
  if (!(rtol > 0.0) || maxit < 1)
    return fail(W3D_ERR_ARG, "w3d_solve_bicgstab: rtol > 0 and maxit >= 1");
  HIPCHK(hipSetDevice(c->device));
  const int n = c->neqns;
  if (!c->d_bicg)
    return fail(W3D_ERR_ARG, "w3d_solve_bicgstab: no workspace (assemble "
                             "the CSR first)");
  double* d = c->d_bicg;
  int rc;
  double* d_b = d;
  double* d_x = d + n;
  HIPCHK(hipMemcpyAsync(d_b, rhs, 8 * (size_t)n, hipMemcpyHostToDevice,
                        c->stream));
  int it = 0;
  double rr = 0.0;
  rc = bicgstab(n, c->groups(), c->d_csr_val, d_b, d_x, d + 2 * (int64_t)n,
                rtol, maxit, &it, &rr, c->h_poll, c->poll_ev, c->stream);
  if (hipMemcpyAsync(x, d_x, 8 * (size_t)n, hipMemcpyDeviceToHost,
                     c->stream) != hipSuccess ||
      hipStreamSynchronize(c->stream) != hipSuccess)
    rc = W3D_ERR_DEVICE;
  if (iters) *iters = it;
  if (relres) *relres = rr;
  if (rc == W3D_ERR_NUMERIC)
    return fail(rc, "w3d_solve_bicgstab: no convergence in " +
                        std::to_string(it) +
                        " iterations or a breakdown (relres " +
                        std::to_string(rr) + ")");
  if (rc) return fail(rc, "w3d_solve_bicgstab: device failure");
  return W3D_OK;
}

int w3d_get_block_ek_full(const w3d_ctx* c, int32_t blk, double* out,
                          int64_t n_out) {
  if (!c || blk < 1 || blk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_get_block_ek_full: block");
  if (!c->asym_tangent)
    return fail(W3D_ERR_ARG, "w3d_get_block_ek_full: no full Ke");
  const BlockDesc& B = c->blocks[blk - 1];
  const int64_t n = (int64_t)B.span * B.totdof * B.totdof;
  if (!out || n_out < n)
    return fail(W3D_ERR_ARG, "w3d_get_block_ek_full: output too small");
  int64_t off = 0;
  for (int b = 0; b < blk - 1; ++b)
    off += (int64_t)c->blocks[b].span * c->blocks[b].totdof *
           c->blocks[b].totdof;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipMemcpy(out, c->d_ekf + off, 8 * (size_t)n, hipMemcpyDeviceToHost));
  return W3D_OK;
}

int w3d_assemble_vss_dev(w3d_ctx* c, double* d_k_diag, double* d_k_coeffs) {
  if (!c || !c->asm_ready) return fail(W3D_ERR_ARG, "w3d_assemble: no pattern");
  if (c->asym)
    return fail(W3D_ERR_ARG, "w3d_assemble_vss: asymmetric assembly is on");
  if (c->tangent_precision < 0)
    return fail(W3D_ERR_ARG, "w3d_assemble: no tangent computed");
  if (!d_k_diag || (!d_k_coeffs && c->ncoeff))
    return fail(W3D_ERR_ARG, "w3d_assemble_vss_dev: null output");
  HIPCHK(hipSetDevice(c->device));
  prof_begin(c, W3D_PHASE_ASSEMBLE);
  int rc = c->enqueue_assemble(c->tangent_precision == W3D_FP32, d_k_diag,
                               d_k_coeffs, c->stream);
  prof_end(c, W3D_PHASE_ASSEMBLE);
  if (rc) return fail(rc, "w3d_assemble: kernel launch failed");
  HIPCHK(hipStreamSynchronize(c->stream));
  prof_collect(c);
  return W3D_OK;
}

int w3d_assemble_vss(w3d_ctx* c, double* k_diag, double* k_coeffs) {
  if (!c || !c->asm_ready) return fail(W3D_ERR_ARG, "w3d_assemble: no pattern");
  if (c->asym)
    return fail(W3D_ERR_ARG, "w3d_assemble_vss: asymmetric assembly is on");
  if (c->tangent_precision < 0)
    return fail(W3D_ERR_ARG, "w3d_assemble: no tangent computed");
  HIPCHK(hipSetDevice(c->device));
  prof_begin(c, W3D_PHASE_ASSEMBLE);
  int rc = c->enqueue_assemble(c->tangent_precision == W3D_FP32, c->d_kout,
                               c->d_kout + c->neqns, c->stream);
  prof_end(c, W3D_PHASE_ASSEMBLE);
  if (rc) return fail(rc, "w3d_assemble: kernel launch failed");
  c->assembled += 1;
  if (k_diag)
    HIPCHK(hipMemcpyAsync(k_diag, c->d_kout, c->neqns * sizeof(double),
                          hipMemcpyDeviceToHost, c->stream));
  if (k_coeffs && c->ncoeff)
    HIPCHK(hipMemcpyAsync(k_coeffs, c->d_kout + c->neqns,
                          c->ncoeff * sizeof(double), hipMemcpyDeviceToHost,
                          c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  prof_collect(c);
  return W3D_OK;
}

int w3d_commit_step(w3d_ctx* c) {
  if (!c) return fail(W3D_ERR_ARG, "null context");
  HIPCHK(hipSetDevice(c->device));
  int rc = enqueue_commit(c);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(c->stream));
  return W3D_OK;
}

int w3d_rollback(w3d_ctx* c) {
  if (!c) return fail(W3D_ERR_ARG, "null context");
  HIPCHK(hipSetDevice(c->device));
  int rc = enqueue_rollback(c);
  if (rc) return rc;
  HIPCHK(hipStreamSynchronize(c->stream));
  return W3D_OK;
}

static int state_size(const BlockDesc& B, int which, int64_t* n) {
  int64_t nq = (int64_t)B.span * B.ngp;
  switch (which) {
    case W3D_STRESS_N: case W3D_STRESS_N1: *n = 9 * nq; return 9;
    case W3D_STRAIN_N: case W3D_STRAIN_N1: *n = 6 * nq; return 6;
    case W3D_HIST_N: case W3D_HIST_N1: *n = B.hist * nq; return B.hist;
    case W3D_CEP: *n = 21 * nq; return 21;
    case W3D_ESTIFF: *n = (int64_t)B.utsz * B.span; return 0;
    case W3D_EINFVEC: *n = (int64_t)B.totdof * B.span; return 0;
    case W3D_ELEM_VOL: *n = B.span; return 0;
    case W3D_ROT_N1:
      if (!B.geonl) break;
      *n = 9 * nq;
      return 9;
    default: break;
  }
  *n = 0;
  return -1;
}

int w3d_get_block_state(const w3d_ctx* c, int32_t blk, int32_t which,
                        double* out, int64_t n_out) {
  if (!c || !out || blk < 1 || blk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_get_block_state: bad block");
  const BlockDesc& B = c->blocks[blk - 1];
  int64_t n;
  int nw = state_size(B, which, &n);
  if (nw < 0 || n_out < n)
    return fail(W3D_ERR_ARG, "w3d_get_block_state: selector or size");
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  const int64_t S = B.span, G = B.ngp, SG = S * G;
  std::vector<double> tmp(n);
  const double* src = nullptr;
  switch (which) {
    case W3D_STRESS_N: src = c->d_stress_n + 9 * B.q_off; break;
    case W3D_STRESS_N1: src = c->d_stress_n1 + 9 * B.q_off; break;
    case W3D_STRAIN_N: src = c->d_strain_n + 6 * B.q_off; break;
    case W3D_STRAIN_N1: src = c->d_strain_n1 + 6 * B.q_off; break;
    case W3D_HIST_N: src = c->d_hist_n + B.hist_off; break;
    case W3D_HIST_N1: src = c->d_hist_n1 + B.hist_off; break;
    case W3D_CEP: src = c->d_cep + 21 * B.q_off; break;
    case W3D_EINFVEC: src = c->d_einfvec + B.ifv_off; break;
    case W3D_ELEM_VOL: src = c->d_evol + (B.felem - 1); break;
    case W3D_ROT_N1: src = c->d_rot_n1 + 9 * B.q_off; break;
    default: break;
  }
  if (which == W3D_ESTIFF) {
    if (c->tangent_precision == W3D_FP32) {
      std::vector<float> f(n);
      HIPCHK(hipMemcpy(f.data(), c->d_ek32 + B.ek_off, n * 4,
                       hipMemcpyDeviceToHost));
      for (int64_t k = 0; k < n; ++k) tmp[k] = f[k];
    } else {
      HIPCHK(hipMemcpy(tmp.data(), c->d_ek64 + B.ek_off, n * 8,
                       hipMemcpyDeviceToHost));
    }
    // ranked row-major order -> packed upper column-major (cp(q) + p)
    for (int64_t i = 0; i < S; ++i) {
      int rank[kMaxNodes];
      node_ranks(&c->conn[B.conn_off + i * B.nnode], B.nnode, rank);
      const double* src = tmp.data() + i * B.utsz;
      double* dst = out + i * B.utsz;
      for (int q = 0; q < B.totdof; ++q)
        for (int p = 0; p <= q; ++p)
          dst[q * (q + 1) / 2 + p] = src[ek_pos(B.nnode, rank, p, q)];
    }
    return W3D_OK;
  }
  HIPCHK(hipMemcpy(tmp.data(), src, n * 8, hipMemcpyDeviceToHost));
  if (which == W3D_ELEM_VOL) {
    std::memcpy(out, tmp.data(), n * 8);
  } else if (which == W3D_EINFVEC) {  // device (i, 3j+c) -> (span, totdof)
    for (int64_t i = 0; i < S; ++i)
      for (int64_t j = 0; j < B.nnode; ++j)
        for (int64_t cc = 0; cc < 3; ++cc)
          out[(cc * B.nnode + j) * S + i] = tmp[i * B.totdof + 3 * j + cc];
  } else if (which == W3D_CEP) {  // device (k, i, g) -> (21, span, ngp)
    for (int64_t k = 0; k < 21; ++k)
      for (int64_t i = 0; i < S; ++i)
        for (int64_t g = 0; g < G; ++g)
          out[(g * S + i) * 21 + k] = tmp[k * SG + i * G + g];
  } else {  // device (k, i, g) -> (nw, ngp, span)
    for (int64_t k = 0; k < nw; ++k)
      for (int64_t i = 0; i < S; ++i)
        for (int64_t g = 0; g < G; ++g)
          out[(i * G + g) * nw + k] = tmp[k * SG + i * G + g];
  }
  return W3D_OK;
}

int w3d_set_block_state(w3d_ctx* c, int32_t blk, int32_t which,
                        const double* in, int64_t n_in) {
  if (!c || !in || blk < 1 || blk > c->nelblk)
    return fail(W3D_ERR_ARG, "w3d_set_block_state: bad block");
  if (which != W3D_STRESS_N && which != W3D_STRAIN_N && which != W3D_HIST_N)
    return fail(W3D_ERR_ARG, "w3d_set_block_state: selector");
  const BlockDesc& B = c->blocks[blk - 1];
  int64_t n;
  int nw = state_size(B, which, &n);
  if (n_in < n) return fail(W3D_ERR_ARG, "w3d_set_block_state: size");
  const int64_t S = B.span, G = B.ngp, SG = S * G;
  std::vector<double> tmp(n);
  for (int64_t k = 0; k < nw; ++k)
    for (int64_t i = 0; i < S; ++i)
      for (int64_t g = 0; g < G; ++g)
        tmp[k * SG + i * G + g] = in[(i * G + g) * nw + k];
  double* dst = which == W3D_STRESS_N   ? c->d_stress_n + 9 * B.q_off
                : which == W3D_STRAIN_N ? c->d_strain_n + 6 * B.q_off
                                        : c->d_hist_n + B.hist_off;
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  HIPCHK(hipMemcpy(dst, tmp.data(), n * 8, hipMemcpyHostToDevice));
  return W3D_OK;
}

int w3d_solve_pcg_dev(w3d_ctx* c, const double* d_k_diag,
                      const double* d_k_coeffs, const double* d_rhs,
                      double* d_x, double rtol, int32_t maxit, int32_t* iters,
                      double* relres) {
  if (!c || !c->d_csr_rp) return fail(W3D_ERR_ARG, "w3d_solve_pcg: no pattern");
  if (!d_k_diag || !d_rhs || !d_x || (!d_k_coeffs && c->ncoeff))
    return fail(W3D_ERR_ARG, "w3d_solve_pcg_dev: null argument");
  if (!(rtol > 0.0) || maxit < 1)
    return fail(W3D_ERR_ARG, "w3d_solve_pcg: rtol > 0 and maxit >= 1");
  HIPCHK(hipSetDevice(c->device));
  return pcg_impl(c, d_k_diag, d_k_coeffs, d_rhs, d_x, rtol, maxit, iters,
                  relres, c->d_pcg,
                  c->d_pcg + kPcgVectors * (int64_t)c->neqns);
}

int w3d_solve_pcg_static(w3d_ctx* c, const double* d_k_diag,
                         const double* d_k_coeffs, const double* d_rhs,
                         double* d_x, double rtol, int32_t maxit,
                         int32_t* iters, double* relres) {
  if (!c || !c->d_csr_rp)
    return fail(W3D_ERR_ARG, "w3d_solve_pcg_static: no pattern");
  if (!d_k_diag || !d_rhs || !d_x || (!d_k_coeffs && c->ncoeff))
    return fail(W3D_ERR_ARG, "w3d_solve_pcg_static: null argument");
  if (!(rtol > 0.0) || maxit < 1)
    return fail(W3D_ERR_ARG, "w3d_solve_pcg_static: rtol > 0 and maxit >= 1");
  if (c->neqns > w3d::kStaticMaxEq)
    return fail(W3D_ERR_ARG,
                "w3d_solve_pcg_static: " + std::to_string(c->neqns) +
                    " equations, more than the static work memory's " +
                    std::to_string(w3d::kStaticMaxEq));
  HIPCHK(hipSetDevice(c->device));
  double* work = nullptr;
  int rc = w3d::solver_static_scratch(c->device, &work);
  if (rc) return fail(rc, "w3d_solve_pcg_static: static work memory");
  return pcg_impl(c, d_k_diag, d_k_coeffs, d_rhs, d_x, rtol, maxit, iters,
                  relres, work,
                  work + kPcgVectors * (int64_t)w3d::kStaticMaxEq);
}

int w3d_solve_pcg(w3d_ctx* c, const double* rhs, double* x, double rtol,
                  int32_t maxit, int32_t* iters, double* relres) {
  if (!c || !c->d_csr_rp) return fail(W3D_ERR_ARG, "w3d_solve_pcg: no pattern");
  if (!c->assembled)
    return fail(W3D_ERR_ARG, "w3d_solve_pcg: no w3d_assemble_vss since the "
                             "pattern");
  if (!rhs || !x) return fail(W3D_ERR_ARG, "w3d_solve_pcg: null argument");
  if (!(rtol > 0.0) || maxit < 1)
    return fail(W3D_ERR_ARG, "w3d_solve_pcg: rtol > 0 and maxit >= 1");
  HIPCHK(hipSetDevice(c->device));
  const int n = c->neqns;
  double* b = c->d_pcg + kPcgVectors * (int64_t)n + kPcgTail;
  double* xd = b + n;
  HIPCHK(hipMemcpyAsync(b, rhs, n * sizeof(double), hipMemcpyHostToDevice,
                        c->stream));
  HIPCHK(hipMemcpyAsync(xd, x, n * sizeof(double), hipMemcpyHostToDevice,
                        c->stream));
  int rc = pcg_impl(c, c->d_kout, c->d_kout + n, b, xd, rtol, maxit, iters,
                    relres, c->d_pcg, c->d_pcg + kPcgVectors * (int64_t)n);
  if (rc < 0 && rc != W3D_ERR_NUMERIC) return rc;
  HIPCHK(hipMemcpyAsync(x, xd, n * sizeof(double), hipMemcpyDeviceToHost,
                        c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  return rc;
}

int w3d_set_time_increment(w3d_ctx* c, double dt) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_set_time_increment: null context");
  if (!(dt > 0.0))
    return fail(W3D_ERR_ARG, "w3d_set_time_increment: dt must be > 0");
  c->dt = dt;
  return W3D_OK;
}

int w3d_set_temperatures(w3d_ctx* c, const double* temper_nodes,
                         const double* dtemp_nodes, const double* temper_elems,
                         const double* dtemp_elems, int32_t incremental) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_set_temperatures: null context");
  const int64_t nn = c->nonode, ne = c->noelem;
  std::vector<double> h(2 * (nn + ne), 0.0);
  if (temper_nodes) std::memcpy(h.data(), temper_nodes, nn * 8);
  if (dtemp_nodes) std::memcpy(h.data() + nn, dtemp_nodes, nn * 8);
  if (temper_elems) std::memcpy(h.data() + 2 * nn, temper_elems, ne * 8);
  if (dtemp_elems) std::memcpy(h.data() + 2 * nn + ne, dtemp_elems, ne * 8);
  HIPCHK(hipSetDevice(c->device));
  // ordered after the work already queued on the context's stream
  HIPCHK(hipStreamSynchronize(c->stream));
  const bool fresh = !c->d_temps;
  if (fresh) {
    int rc = dalloc(&c->d_temps, (int64_t)h.size());
    if (rc) return rc;
  }
  HIPCHK(hipMemcpy(c->d_temps, h.data(), h.size() * 8,
                   hipMemcpyHostToDevice));
  // captured iterations hold the temperature pointer and flag by value
  if (fresh || c->temps_incr != (incremental != 0)) {
    for (auto& g : c->graphs) (void)hipGraphExecDestroy(g.exec);
    c->graphs.clear();
  }
  c->temps_incr = incremental != 0;
  return W3D_OK;
}

int w3d_set_profiling(w3d_ctx* c, int32_t on) {
  if (!c) return fail(W3D_ERR_ARG, "null context");
  HIPCHK(hipSetDevice(c->device));
  if (on && !c->ev_a[0][0])
    for (int ph = 0; ph < W3D_NUM_PHASES; ++ph) {
      for (int k = 0; k < 2; ++k) {
        HIPCHK(hipEventCreate(&c->ev_a[ph][k]));
        HIPCHK(hipEventCreate(&c->ev_b[ph][k]));
      }
    }
  c->profiling = on != 0;
  return W3D_OK;
}

int w3d_get_phase_time(const w3d_ctx* c, int32_t phase, int64_t* launches,
                       double* total_ms) {
  if (!c || phase < 0 || phase >= W3D_NUM_PHASES)
    return fail(W3D_ERR_ARG, "w3d_get_phase_time: phase");
  if (launches) *launches = c->prof_n[phase];
  if (total_ms) *total_ms = c->prof_ms[phase];
  return W3D_OK;
}

int w3d_reset_phase_times(w3d_ctx* c) {
  if (!c) return fail(W3D_ERR_ARG, "null context");
  for (int ph = 0; ph < W3D_NUM_PHASES; ++ph) {
    c->prof_n[ph] = 0;
    c->prof_ms[ph] = 0.0;
  }
  return W3D_OK;
}

int w3d_synchronize(w3d_ctx* c) {
  if (!c) return fail(W3D_ERR_ARG, "null context");
  HIPCHK(hipSetDevice(c->device));
  HIPCHK(hipStreamSynchronize(c->stream));
  return W3D_OK;
}

int w3d_iteration_dev(w3d_ctx* c, int32_t step, int32_t iter,
                      int32_t extrapolated, const double* d_u,
                      const double* d_du, double* d_ifv, int32_t precision,
                      double* d_k_diag, double* d_k_coeffs, double* energy,
                      double* plastic_work) {
  if (!c || !d_du || !d_ifv)
    return fail(W3D_ERR_ARG, "w3d_iteration_dev: null argument");
  if (c->asym)
    return fail(W3D_ERR_UNSUPPORTED,
                "w3d_iteration_dev: asymmetric assembly (symmetric VSS only)");
  if (step < 1 || iter < 0)
    return fail(W3D_ERR_ARG, "w3d_iteration_dev: step/iter");
  if (precision != W3D_FP64 && precision != W3D_FP32)
    return fail(W3D_ERR_ARG, "w3d_iteration_dev: precision");
  if (!c->asm_ready) return fail(W3D_ERR_ARG, "w3d_iteration_dev: no pattern");
  if (!d_k_diag || (!d_k_coeffs && c->ncoeff))
    return fail(W3D_ERR_ARG, "w3d_iteration_dev: null matrix output");
  HIPCHK(hipSetDevice(c->device));
  // the kernels see the step and the iteration only through these
  // predicates: one graph per (step 1?, iteration 0?, extrapolated,
  // precision, energy sums) and per set of caller buffers and dt
  const int step_c = step == 1 ? 1 : 2, iter_c = iter == 0 ? 0 : 1;
  const bool sums = energy || plastic_work;
  const int key[5] = {step_c, iter_c, extrapolated ? 1 : 0, precision,
                      sums ? 1 : 0};
  const void* ptr[5] = {d_u, d_du, d_ifv, d_k_diag, d_k_coeffs};
  w3d_ctx::GraphEntry* ge = nullptr;
  for (auto& g : c->graphs)
    if (!std::memcmp(g.key, key, sizeof key) &&
        !std::memcmp(g.ptr, ptr, sizeof ptr) && g.dt == c->dt)
      ge = &g;
  if (!ge) {
    if (c->graphs.size() >= 8) {
      (void)hipGraphExecDestroy(c->graphs.front().exec);
      c->graphs.erase(c->graphs.begin());
    }
    RecoverLists L;
    int rc = recover_lists(c, L);  // the resident lists
    if (rc) return rc;
    L.host = c->h_rec;
    HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    c->capturing = true;
    rc = enqueue_recover(c, L, step_c, iter_c, extrapolated ? 1 : 0, d_u, d_du,
                         d_ifv, sums, 1, c->nelblk);
    if (!rc)
      rc = launch_tangent_mfma(c->dev(), c->d_work_tan, c->tan_groups,
                               c->tan_start, c->tan_count, precision,
                               c->stream);
    if (!rc)
      rc = c->enqueue_assemble(precision == W3D_FP32, d_k_diag, d_k_coeffs,
                               c->stream);
    c->capturing = false;
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(c->stream, &graph);
    if (rc || e != hipSuccess) {
      if (graph) (void)hipGraphDestroy(graph);
      return rc ? rc : fail(W3D_ERR_DEVICE, "w3d_iteration_dev: capture");
    }
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess)
      return fail(W3D_ERR_DEVICE, std::string("hipGraphInstantiate: ") +
                                      hipGetErrorString(e));
    w3d_ctx::GraphEntry g;
    std::memcpy(g.key, key, sizeof key);
    std::memcpy(g.ptr, ptr, sizeof ptr);
    g.dt = c->dt;
    g.exec = exec;
    c->graphs.push_back(g);
    ge = &c->graphs.back();
  }
  HIPCHK(hipGraphLaunch(ge->exec, c->stream));
  c->tangent_precision = precision;
  c->assembled += 1;
  return finish_recover(c, step, iter, energy, plastic_work);
}

int w3d_autotune(w3d_ctx* c, int32_t precision, int32_t* choices,
                 int32_t capacity, int32_t* n_choices) {
  if (!c) return fail(W3D_ERR_ARG, "w3d_autotune: null context");
  if (precision != W3D_FP64 && precision != W3D_FP32)
    return fail(W3D_ERR_ARG, "w3d_autotune: precision");
  HIPCHK(hipSetDevice(c->device));
  hipEvent_t ea, eb;
  HIPCHK(hipEventCreate(&ea));
  HIPCHK(hipEventCreate(&eb));
  DevModel M = c->dev();
  std::vector<int32_t> out;
  int rc = W3D_OK;
  // tangent: per kernel group the work-item size, in elements, with the
  // shortest launch (the mean of three, the shortest of three such, after
  // one untimed launch: of single means a small model's scatter by more than
  // its sizes differ); 0 is build_work's own
  auto set_chunk = [&](int key, int chunk) {
    auto& tc = c->tan_chunk;
    tc.erase(std::remove_if(tc.begin(), tc.end(),
                            [&](const auto& kc) { return kc.first == key; }),
             tc.end());
    if (chunk > 0) tc.push_back({key, chunk});
  };
  const std::vector<int> groups = c->tan_groups;
  for (int key : groups) {
    int best = 0;
    float best_ms = 0.0f;
    for (int chunk : {0, 8, 16, 32, 64}) {
      set_chunk(key, chunk);
      std::vector<WorkItem> items;
      std::vector<int> g, st, cnt;
      build_work(c, true, items, g, st, cnt);
      size_t k = 0;
      while (k < g.size() && g[k] != key) ++k;
      if (k == g.size()) continue;
      std::vector<WorkItem> mine(items.begin() + st[k],
                                 items.begin() + st[k] + cnt[k]);
      WorkItem* d = nullptr;
      if ((rc = upload(&d, mine))) break;
      const std::vector<int> gg{key}, ss{0}, nn{cnt[k]};
      rc = launch_tangent_mfma(M, d, gg, ss, nn, precision, c->stream);
      float ms = 0.0f;
      for (int m = 0; m < 3 && !rc; ++m) {
        (void)hipEventRecord(ea, c->stream);
        for (int r = 0; r < 3 && !rc; ++r)
          rc = launch_tangent_mfma(M, d, gg, ss, nn, precision, c->stream);
        (void)hipEventRecord(eb, c->stream);
        (void)hipStreamSynchronize(c->stream);
        float t = 0.0f;
        (void)hipEventElapsedTime(&t, ea, eb);
        ms = m == 0 || t < ms ? t : ms;
      }
      dfree(d);
      if (rc) break;
      if (!chunk || ms < best_ms) {
        best = chunk;
        best_ms = ms;
      }
    }
    set_chunk(key, rc ? 0 : best);
    if (rc) break;
    if (!best) continue;
    out.push_back(key);
    out.push_back(best);
  }
  // persistent mm10: workgroups per compute unit (after a recovery the
  // increments are in place; the kernel rewrites the same outputs from the
  // same inputs)
  if (!rc && c->has_mm10 && c->n_work_mm10 > 0) {
    const int iter0_off = 0;
    int best = c->mm10_grid;
    float best_ms = 0.0f;
    for (int per_cu : {2, 4, 8}) {
      const int grid = per_cu * std::max(c->n_cu, 1);
      rc = launch_mm10(M, c->d_work_mm10, c->n_work_mm10, c->d_counter, grid,
                       c->last_step, iter0_off, c->stream);
      (void)hipEventRecord(ea, c->stream);
      for (int r = 0; r < 2 && !rc; ++r)
        rc = launch_mm10(M, c->d_work_mm10, c->n_work_mm10, c->d_counter,
                         grid, c->last_step, iter0_off, c->stream);
      (void)hipEventRecord(eb, c->stream);
      (void)hipStreamSynchronize(c->stream);
      if (rc) break;
      float ms = 0.0f;
      (void)hipEventElapsedTime(&ms, ea, eb);
      if (per_cu == 2 || ms < best_ms) {
        best = grid;
        best_ms = ms;
      }
    }
    c->mm10_grid = best;
    out.push_back(-1);
    out.push_back(best);
  }
  (void)hipEventDestroy(ea);
  (void)hipEventDestroy(eb);
  if (rc) return fail(rc, "w3d_autotune: launch failed");
  // the tangent work list with the chosen sizes; captured iterations are
  // stale
  std::vector<WorkItem> items;
  build_work(c, true, items, c->tan_groups, c->tan_start, c->tan_count);
  dfree(c->d_work_tan);
  if ((rc = upload(&c->d_work_tan, items))) return rc;
  build_runs(c);
  for (auto& g : c->graphs) (void)hipGraphExecDestroy(g.exec);
  c->graphs.clear();
  if (choices)
    for (int32_t k = 0; k < capacity && k < (int32_t)out.size(); ++k)
      choices[k] = out[k];
  if (n_choices) *n_choices = (int32_t)out.size();
  return W3D_OK;
}

}  // extern "C"
