// Launches of the bonded terms and the 1-4 / exclusion pairs (bodies in
// bonded_terms.hpp) that do not ride in the pair kernel's: energy and virial
// calls, forked force calls from 10,000 atoms, and fused batches.
#include "bonded_terms.hpp"

namespace apo {

// Each list alone is latency-bound and too small to fill the chip: side by
// side in one launch they take what the longer one takes.
template <typename CT, bool CALC_E, bool CALC_V>
__global__ __launch_bounds__(256) void k_bonded14(Bonded14<CT> B, double *__restrict__ part14,
                                                  const PairConsts<double> PE,
                                                  const double2 *__restrict__ tab14_e,
                                                  double *__restrict__ partb) {
  bonded14_body<CT, CALC_E, CALC_V, 256>(blockIdx.x, B, part14, PE, tab14_e, partb);
}

struct BondedBatchArgs {
  BondedArgs a;
  unsigned long long *f;
};
struct P14BatchArgs {
  P14Args a;
  PairConsts<float> P;
  const float2 *tab14;
  unsigned long long *f;
};
__global__ __launch_bounds__(256) void kb_bonded(const BondedBatchArgs *__restrict__ tab,
                                                 const int *__restrict__ bstart, int nsys) {
  const int s = batch_system(bstart, nsys);
  const BondedBatchArgs &a = tab[s];
  bonded_body<float, false, false, 256>(blockIdx.x - bstart[s], a.a, a.f, nullptr);
}
__global__ __launch_bounds__(256) void kb_pairs14(const P14BatchArgs *__restrict__ tab,
                                                  const int *__restrict__ bstart, int nsys) {
  const int s = batch_system(bstart, nsys);
  const P14BatchArgs &a = tab[s];
  const PairConsts<double> no_energy{};
  pairs14_body<float, false, false, 256>(blockIdx.x - bstart[s], a.a, a.P, a.tab14, a.f, nullptr,
                                    no_energy, nullptr);
}


template <typename CT, typename F>
static void dispatch_ev(bool E, bool V, F &&fn) {
  if (E && V) fn(std::integral_constant<int, 3>());
  else if (E) fn(std::integral_constant<int, 1>());
  else if (V) fn(std::integral_constant<int, 2>());
  else fn(std::integral_constant<int, 0>());
}

void bonded_launch(NbSystem &S, const float4 *x, int64_t *force, int stride, bool E, bool V,
                   bool pairs14, bool bonded, hipStream_t s) {
  double *part14 = S.parts_ptr() + S.part.p14_off, *partb = S.parts_ptr() + S.part.bond_off;
  auto run = [&](auto ct, auto ev) {
    using CT = decltype(ct);
    constexpr int m = decltype(ev)::value;
    const Bonded14<CT> B = bonded14_args<CT>(S, x, force, stride, pairs14, bonded, 256);
    if (B.n14 + B.nb == 0) return;
    k_bonded14<CT, (m & 1) != 0, (m & 2) != 0>
        <<<B.n14 + B.nb, 256, 0, s>>>(B, part14, S.pc_d, S.vdwtab14_d.get(), partb);
    APO_LAUNCH_CHECK();
  };
  auto go = [&](auto ev) {
    if (S.precision == 1) run(double(), ev);
    else run(float(), ev);
  };
  dispatch_ev<float>(E, V, go);
}

// ---- fused launches over several systems (mixed precision, no energy) ------
struct BondedBatch {
  BatchLaunch<BondedBatchArgs> bonded;
  BatchLaunch<P14BatchArgs> p14;
};
BondedBatch *bonded_batch_create() { return new BondedBatch(); }
void bonded_batch_destroy(BondedBatch *b) { delete b; }
void bonded_batch_clear(BondedBatch &b) {
  b.bonded.clear();
  b.p14.clear();
}
void bonded_batch_add(BondedBatch &b, NbSystem &S, const float4 *x, int64_t *force, int stride) {
  if (S.precision != 0) throw InvalidArgument("fused batches run the mixed-precision path");
  auto *f = reinterpret_cast<unsigned long long *>(force);
  const int nt = S.nbond + S.nub + S.nangle + S.ndihe + S.nimdihe;
  if (nt > 0)
    b.bonded.add(BondedBatchArgs{BondedArgs{x, S.bonds.get(), S.ureyb.get(), S.angles.get(),
                                            S.dihe.get(), S.imdihe.get(), S.nbond, S.nub,
                                            S.nangle, S.ndihe, S.nimdihe, stride},
                                 f},
                 S.part.bond_n);
  if (S.nin14 + S.nex14 > 0)
    b.p14.add(P14BatchArgs{P14Args{x, S.vdwtype.get(), S.in14.get(), S.ex14.get(), S.nin14,
                                   S.nex14, stride, S.ntypes, S.e14fac},
                           S.pc_f, S.vdwtab14.get(), f},
              S.part.p14_n);
}
void bonded_batch_upload(BondedBatch &b, hipStream_t s) {
  b.bonded.upload(s);
  b.p14.upload(s);
}
void bonded_batch_launch(BondedBatch &b, hipStream_t s) {
  if (b.bonded.nsys())
    kb_bonded<<<b.bonded.blocks(), 256, 0, s>>>(b.bonded.d_args.get(), b.bonded.d_start.get(),
                                                b.bonded.nsys());
  if (b.p14.nsys())
    kb_pairs14<<<b.p14.blocks(), 256, 0, s>>>(b.p14.d_args.get(), b.p14.d_start.get(),
                                              b.p14.nsys());
  APO_LAUNCH_CHECK();
}

}  // namespace apo
