// Order of the memory requests of the 128 x 128 kernel (mx_gemm_t128.hip) and the counted waits that follow from it.
// Plain C++ without device code, so that the rules can be checked on the host.
//
// A wave requests stages of TL loads each, NS stages ahead, and one load of scales per K-quad (SPQ stages).  Its loads
// complete in the order of the requests, so "at most n outstanding" means that all but the n youngest are in LDS.
//   prologue: stages 0 .. NS - 1, the scales of a quad in front of its first stage; wait; stage 0 and the scales of quad 0
//             are read
//   stage s:  wait; barrier; at the first stage of quad Q the scales of quad Q + SD are requested, then stage s + NS; stage
//             s + 1 is read, at the last stage of quad Q also the scales of quad Q + 1
// The prologue's order is the one that the stages continue.  (All scales ahead of the stages, it would leave one load
// fewer behind stage 1 than the stages' count assumes.)
// Scales at any byte come through registers: a quad's kAnyLoads loads are requested into them where the loads of scales above
// have their place, one quad ahead, and go to LDS a quad later, behind the barrier of that quad's first stage; all waves read them
// at its last stage.  (The register contents are waited for by their own use.)
#pragma once

namespace mx {

template <int NS_, int SPQ_, int TL_>
struct T128Schedule {
  static constexpr int NS = NS_, SPQ = SPQ_, TL = TL_;
  static constexpr int SD = (NS + SPQ - 1) / SPQ;          // quads of scales in flight
  // scales that the prologue requests in front of stage k: those of quad k / SPQ
  static constexpr bool prologue_scales(int k) { return k % SPQ == 0; }
  // behind stage 0: the other stages and the scales requested between them
  static constexpr int prologue_wait() { return (NS - 1) * TL + SD - 1; }
  // behind stage s + 1, t = s % SPQ: NS - 2 stages, and the scales that the stages of those requests asked for
  static constexpr int stage_wait(int t) {
    int n = (NS - 2) * TL;
    for (int back = 1; back <= NS - 2; ++back) n += (t + SPQ * NS - back) % SPQ == 0;
    return n;
  }
  // Scales that come through registers are loads whose place and number the waits leave out: of the stages' loads alone,
  // NS - 1 (NS - 2) stages are behind stage 0 (s + 1), so a wait for all but these is never too short.
  static constexpr int kAnyLoads = 5;
  static constexpr int any_prologue_wait() { return (NS - 1) * TL; }
  static constexpr int any_stage_wait() { return (NS - 2) * TL; }
};

// Whether 64 x 64 tiles with eight stages in flight and scales at any byte send a stage's requests between its MFMAs: for short K only.
// (Why that costs them beyond, and neither packed nor aligned scales, is not measured.)
// us, behind the barrier | between the MFMAs, K in one range: FP8 500 x 1500 and 900 x 900, K = 2048 8.5 | 8.4, 8.7 | 8.4, 3072 (E5M2) 10.8 | 10.5,
// 11.1 | 10.7, 4096 12.8 | 12.5, 13.4 | 13.7, 5120 15.5 | 15.4, 16.5 | 17.0, 7168 21.1 | 21.8, 21.3 | 22.0, 14336 36.4 | 38.8, 37.0 | 39.2; FP4
// weights 4096 12.0 | 11.9, 12.0 | 11.8, 5120 13.7 | 13.6, 14.3 | 15.4, 8192 19.9 | 21.9, 20.8 | 22.6; FP4 x FP4 4096 9.8 | 9.6, 9.8 | 9.6, 5120 11.1 |
// 10.8, 10.9 | 11.0, 7168 13.5 | 13.4, 14.0 | 15.3, 14336 25.2 | 27.9, 25.7 | 28.3.  With four stages in flight, two workgroups per CU, level: 1000 x
// 1900 FP8 4096 20.4 | 19.5, 8192 33.3 | 33.6.
inline bool t128_any_spread(int K, int splits, int ksteps_per_stage) { return K <= (ksteps_per_stage == 2 ? 5120 : 4096) * (splits > 1 ? splits : 1); }

// First stage of a product of `stages` stages at which something is read that the waits do not cover, -1 if none.  -2: the
// first reads, behind the prologue.  `scales_first`: a prologue that requests all its scales ahead of the stages.
template <class S>
constexpr int t128_uncovered(int stages, bool scales_first = false, int prologue_wait = S::prologue_wait()) {
  constexpr int kMax = 64;
  int stage_end[kMax] = {}, scales_end[kMax] = {}, issued = 0;   // loads requested up to and with the item's last one
  if (stages + S::NS > kMax) return -3;
  if (scales_first)
    for (int q = 0; q < S::SD; ++q) scales_end[q] = ++issued;
  for (int k = 0; k < S::NS; ++k) {
    if (!scales_first && S::prologue_scales(k)) scales_end[k / S::SPQ] = ++issued;
    stage_end[k] = issued += S::TL;
  }
  if (stage_end[0] > issued - prologue_wait || scales_end[0] > issued - prologue_wait) return -2;
  for (int s = 0; s < stages; ++s) {
    const int t = s % S::SPQ, quad = s / S::SPQ, landed = issued - S::stage_wait(t);
    if (stage_end[s + 1] == 0 || stage_end[s + 1] > landed) return s;
    if (t == S::SPQ - 1 && (scales_end[quad + 1] == 0 || scales_end[quad + 1] > landed)) return s;
    if (t == 0) scales_end[quad + S::SD] = ++issued;
    stage_end[s + S::NS] = issued += S::TL;
  }
  return -1;
}

// The same for scales at any byte; -4: a wave reads a quad's scales that another may not have written yet.  `loads`: of a quad's kAnyLoads
// those still among the requests that a wait counts; `ahead`: of the first quad's those that lie ahead of stage 0.
template <class S>
constexpr int t128_any_uncovered(int stages, int loads = S::kAnyLoads, int ahead = S::kAnyLoads, int prologue_wait = S::any_prologue_wait(),
                                 int stage_wait = S::any_stage_wait()) {
  constexpr int kMax = 64;
  int stage_end[kMax] = {}, issued = 0, barriers = 0;
  int written[kMax] = {};                                // barriers ahead of it, + 1
  if (stages + S::NS > kMax) return -3;
  if (ahead > loads) ahead = loads;
  issued += ahead;
  for (int k = 0; k < S::NS; ++k) {
    stage_end[k] = issued += S::TL;
    if (k == 0) issued += loads - ahead;
  }
  if (stage_end[0] > issued - prologue_wait) return -2;
  written[0] = barriers + 1;
  issued += loads;                                       // quad 1
  ++barriers;                                            // quad 0 is read behind it
  for (int s = 0; s < stages; ++s) {
    const int t = s % S::SPQ, quad = s / S::SPQ;
    if (stage_end[s + 1] == 0 || stage_end[s + 1] > issued - stage_wait) return s;
    ++barriers;
    if (t == 0) {
      written[quad + 1] = barriers + 1;
      issued += loads;                                   // quad + 2
    }
    stage_end[s + S::NS] = issued += S::TL;
    if (t == S::SPQ - 1 && written[quad + 1] >= barriers + 1) return -4;
  }
  return -1;
}

template <class S>
constexpr bool t128_covered() {
  for (int stages = 1; stages <= 24; ++stages) {
    if (t128_uncovered<S>(stages) != -1) return false;
    for (int loads = 0; loads <= S::kAnyLoads; ++loads)
      for (int ahead = 0; ahead <= loads; ++ahead)
        if (t128_any_uncovered<S>(stages, loads, ahead) != -1) return false;
  }
  return true;
}

}  // namespace mx
