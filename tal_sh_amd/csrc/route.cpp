// Choice between the ways a contraction can run.
#include "route.hpp"

#include <algorithm>

namespace tal {

// Straight from the tensors where the transposes would cost more than the
// reads in place do.  Measured: a K step that walks runs of k costs up to 5 % of
// a product in a kind's largest tiles, 128 x 128 real (R8 9216^3: 21.99 -> 22.66
// ms) and 64 x 64 complex (1600^3 by copies of both operands and in place: C8
// 552 -> 517 us, C4 291 -> 282; 4624 x 4624 by 4096 10,700 -> 10,460 and 5,160
// -> 5,180), and about a quarter in smaller ones (R8 1024^3: 41 -> 50 us), there
// with runs of any length, as offsets then come from tables (runs of 20-24 by
// copies and in place: R8 930 x 957 by 616 60 -> 56 us, 1480 x 1189 by 280 55 ->
// 51, C4 311 x 336 by 600 40 -> 34, C8 550 x 552 by 420 64 -> 65; runs of 32, R8
// 1024^3, 72 -> 79); in 128 x 128 tiles short runs, and any runs by table, cost
// 40 % (complex tiles are held to the same line, though runs of 16 cost them
// little: C8 1600^3 549 by copies, 518 in place); D written 8 bytes apart, about
// four times its bytes.
// A transpose moves 4.6 TB/s and takes about 4 us beside that.
Route contract_route(const ContractPlan &plan, int dk, DirectChooser choose) {
  DirectVariant v;
  if (plan.direct_ok && direct_addressable(plan.direct, dk, &v) && v.mode < 3) {
    const DirectForm &f = plan.direct;
    const int esz = direct_elem(dk);
    const bool d_copy = plan.d_transpose && !plan.mat_d_in_place;
    if (!plan.a.transpose && !plan.b.transpose && !d_copy) return kRouteCopies;  // nothing to copy
    const double avol = (double)f.avol * esz, bvol = (double)f.bvol * esz;
    const double dvol = (double)f.M * (double)f.N * (double)f.batch * esz;
    const bool ta = plan.swap ? plan.b.transpose : plan.a.transpose, tb = plan.swap ? plan.a.transpose : plan.b.transpose;
    const double copies =
        (2 * ((ta ? avol : 0) + (tb ? bvol : 0) + (d_copy ? dvol : 0))) / 4.6e6 + ((ta || tb) ? 4 : 0) + (d_copy ? 4 : 0);
    const DirectChoice c = choose(dk, f.M, f.N, f.K, f.batch);
    const double gemm = c.us;
    double extra = 0;
    if (plan.direct_krun) extra += (c.tile ? 0.25 : plan.direct_krun < 32 || v.mode == 2 ? 0.4 : 0.05) * gemm;
    if (plan.direct_run && plan.direct_run < 8) extra += 0.3 * gemm;
    if (plan.direct_conflict) extra += std::min(avol, bvol) > 4e6 ? 1e9 : 0.5 * gemm;
    if (plan.direct_scatter) extra += 4 * dvol / 4.6e6;
    if (copies > extra) return kRouteDirect;
  }
  return kRouteCopies;
}

}  // namespace tal
