// Orbital-pair tables of the convolution engine (see engine.h).
#include "engine.h"

namespace gmod {

void OrbPairs::from_olist(const int64_t* olist, int Nchi_, int No_) {
  Nchi = Nchi_;
  No = No_;
  ol.resize(Nchi);
  for (int l = 0; l < Nchi; ++l) {
    ol[l] = {(int)olist[l] - 1, (int)olist[l + Nchi] - 1};
    if (ol[l][0] < 0 || ol[l][0] >= No || ol[l][1] < 0 || ol[l][1] >= No)
      throw Error("olist entry outside [1,Norb]");
  }
  // exchange-symmetry partners chi_{1234} = chi*_{4321} (fchi.f90:421-481)
  partner.assign(Nchi * Nchi, {-1, -1});
  psign.assign(Nchi * Nchi, 1.0);
  std::vector<char> cirr(Nchi * Nchi, 0);
  for (int l1 = 0; l1 < Nchi; ++l1)
    for (int m1 = 0; m1 < Nchi; ++m1) {
      bool found = false;
      for (int l2 = 0; l2 < Nchi && !found; ++l2)
        for (int m2 = 0; m2 < Nchi; ++m2) {
          if (ol[l1][0] == ol[m2][1] && ol[l1][1] == ol[m2][0] && ol[m1][0] == ol[l2][1] &&
              ol[m1][1] == ol[l2][0]) {
            partner[m1 + Nchi * l1] = {m2, l2};
            if (!cirr[m2 + Nchi * l2]) cirr[m1 + Nchi * l1] = 1;
            found = true;
            break;
          }
        }
    }
  irr.clear();
  for (int l1 = 0; l1 < Nchi; ++l1)
    for (int m1 = 0; m1 < Nchi; ++m1)
      if (cirr[m1 + Nchi * l1]) irr.push_back({l1, m1});
  const size_t P = (size_t)Nchi * (Nchi + 1) / 2;
  if (irr.size() > P) irr.resize(P);
}

void OrbPairs::from_olist_soc(const int64_t* olist, int Nchi_, int No_, const int64_t* invs, const int64_t* slist) {
  Nchi = Nchi_;
  No = No_;
  soc = true;
  ol.resize(Nchi);
  inv.resize(No);
  spin.resize(No);
  for (int a = 0; a < No; ++a) {
    inv[a] = (int)invs[a] - 1;
    spin[a] = (double)slist[a];
    if (inv[a] < 0 || inv[a] >= No) throw Error("invs entry outside [1,Norb]");
    if (slist[a] != 1 && slist[a] != -1) throw Error("slist entries must be +1 or -1");
  }
  for (int l = 0; l < Nchi; ++l) {
    ol[l] = {(int)olist[l] - 1, (int)olist[l + Nchi] - 1};
    if (ol[l][0] < 0 || ol[l][0] >= No || ol[l][1] < 0 || ol[l][1] >= No)
      throw Error("olist entry outside [1,Norb]");
  }
  // the pair (l, m) and its spin-flipped exchange partner (m2, l2):
  // (l1, l2, m1, m2) = (-m2_2, -m2_1, -l2_2, -l2_1); the first of the two
  // in (l, m) order is the one computed
  partner.assign(Nchi * Nchi, {-1, -1});
  psign.assign(Nchi * Nchi, 1.0);
  std::vector<char> cirr(Nchi * Nchi, 0);
  for (int l1 = 0; l1 < Nchi; ++l1)
    for (int m1 = 0; m1 < Nchi; ++m1) {
      bool found = false;
      for (int l2 = 0; l2 < Nchi && !found; ++l2)
        for (int m2 = 0; m2 < Nchi; ++m2) {
          if (ol[l1][0] == inv[ol[m2][1]] && ol[l1][1] == inv[ol[m2][0]] && ol[m1][0] == inv[ol[l2][1]] &&
              ol[m1][1] == inv[ol[l2][0]]) {
            partner[m1 + Nchi * l1] = {m2, l2};
            if (!cirr[m2 + Nchi * l2]) cirr[m1 + Nchi * l1] = 1;
            found = true;
            break;
          }
        }
      psign[m1 + Nchi * l1] = spin[ol[l1][0]] * spin[ol[l1][1]] * spin[ol[m1][0]] * spin[ol[m1][1]];
    }
  irr.clear();
  for (int l1 = 0; l1 < Nchi; ++l1)
    for (int m1 = 0; m1 < Nchi; ++m1)
      if (cirr[m1 + Nchi * l1]) irr.push_back({l1, m1});
  const size_t P = (size_t)Nchi * (Nchi + 1) / 2;
  if (irr.size() > P) irr.resize(P);
}

void OrbPairs::from_maps(const int32_t* irr_chi, const int32_t* chi_map) {
  const int P = Nchi * (Nchi + 1) / 2;
  irr.resize(P);
  for (int i = 0; i < P; ++i) irr[i] = {irr_chi[i] - 1, irr_chi[i + P] - 1};
  partner.assign(Nchi * Nchi, {-1, -1});
  if (psign.size() != (size_t)Nchi * Nchi) psign.assign(Nchi * Nchi, 1.0);
  for (int l = 0; l < Nchi; ++l)
    for (int m = 0; m < Nchi; ++m)
      partner[m + Nchi * l] = {chi_map[m + Nchi * l] - 1, chi_map[m + Nchi * l + Nchi * Nchi] - 1};
}

}  // namespace gmod
