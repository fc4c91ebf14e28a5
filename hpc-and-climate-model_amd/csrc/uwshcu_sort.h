// uwshcu_sort.h -- S11, the buoyancy sorting (uwshcu.F90:2296-2952), one level at a time.
//
// The sorting runs three times over a column's levels from the release level to the cloud
// top, each time with the last one's cloud-top height.  Its parts are separate members so
// that a lane can go on with another column as soon as its own has ended (sort_kernel).
#ifndef UWSHCU_SORT_H
#define UWSHCU_SORT_H

#include "uwshcu_column.h"

namespace uwshcu {

// Layer k's environment (EnvLevel): its first eight values (lower), the others (upper), or
// all.  From the records where there are any, else from the arrays.
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE EnvLevelOf<D> Column<R, D, ZW, FAST>::env_level_lower(int k) const {
    EnvLevelOf<D> e;
    if constexpr (kRec) {
        const Pair* const r = record(k);
        const Pair p = r[0], q = r[1], s = r[2], t = r[3];
        e.p0 = p.x; e.dp0 = p.y; e.exn0 = q.x; e.thv0bot = q.y; e.thl0 = s.x; e.qt0 = s.y; e.u0 = t.x; e.v0 = t.y;
        return e;
    }
    e.p0 = in(a.p0, k); e.dp0 = in(a.dp0, k); e.exn0 = Ec(A_EXN0, k); e.thv0bot = E(A_THV0BOT, k);
    e.thl0 = E(A_THL0, k); e.qt0 = E(A_QT0, k); e.u0 = in(a.u0, k); e.v0 = in(a.v0, k);
    return e;
}
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE EnvLevelOf<D> Column<R, D, ZW, FAST>::env_level_upper(int k) const {
    EnvLevelOf<D> e;
    if constexpr (kRec) {
        const Pair* const r = record(k);
        const Pair m = r[4], p = r[5], q = r[6], s = r[7], t = r[8];
        e.thv0mid = m.x; e.qs0mid = m.y; e.z0 = p.x; e.thv0top = p.y; e.ssthl = q.x; e.ssqt = q.y;
        e.ssu = s.x; e.ssv = s.y; e.ps0 = t.x; e.exns0 = t.y;
        return e;
    }
    e.z0 = in(a.z0, k); e.thv0top = E(A_THV0TOP, k); e.ssthl = E(A_SSTHL0, k); e.ssqt = E(A_SSQT0, k);
    e.ssu = E(A_SSU0, k); e.ssv = E(A_SSV0, k); e.ps0 = in(a.ps0, k); e.exns0 = Ec(A_EXNS0, k);
    return e;
}
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE EnvLevelOf<D> Column<R, D, ZW, FAST>::env_level(int k) const {
    EnvLevelOf<D> e = env_level_upper(k);
    const EnvLevelOf<D> l = env_level_lower(k);
    e.p0 = l.p0; e.dp0 = l.dp0; e.exn0 = l.exn0; e.thv0bot = l.thv0bot; e.thl0 = l.thl0; e.qt0 = l.qt0;
    e.u0 = l.u0; e.v0 = l.v0;
    return e;
}

template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE void Column<R, D, ZW, FAST>::sort_begin(SortState<R, D>& q, int iter) const {
    q.iter = iter;
    q.scaleh = R(q.cush);
    if (R(q.cush) < R(0)) q.scaleh = R(1000);
    const int krel = q.krel;
    q.kbup = krel;
    q.kpen = krel;
    q.k = krel;
    q.wtw = q.wlcl * q.wlcl;
    const EnvLevelOf<D> e = env_level(krel);
    q.pe = R(0.5) * (q.prel + R(e.ps0));
    q.dpe = q.prel - R(e.ps0);
    q.exe = T.exnf(D(q.pe));          // Exner function of pe, FP64
    q.exne = R(q.exe);
    q.thvebot = q.thv0rel;
    q.pe_tr = q.pe - R(e.p0);
    q.thle = R(e.thl0) + R(e.ssthl) * q.pe_tr;
    q.qte = R(e.qt0) + R(e.ssqt) * q.pe_tr;
    q.ue = R(e.u0) + R(e.ssu) * q.pe_tr;
    q.ve = R(e.v0) + R(e.ssv) * q.pe_tr;
    q.dp0 = e.dp0;
    // tre(m) = tr0(krel,m) + sstr0(krel,m)*(pe - p0(krel)) is recomputed where used
    q.ktr = krel;            // layer whose (tr0, sstr0) define tre, and offset pe_tr
    q.tr_mid = false;        // after the first layer tre = tr0(k) exactly
    sort_release(q);
}

// The plume at the release level, where it starts: from the workspace, or, in the launches
// of a split, from the saved scalars.
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE void Column<R, D, ZW, FAST>::sort_release(SortState<R, D>& q) const {
    if constexpr (kRec) {
        q.thlu = R(rstate(21));
        q.qtu = R(rstate(22));
        q.uu = R(rstate(23));
        q.vu = R(rstate(24));
        q.thvu = R(rstate(25));
        q.wu = R(rstate(26));
        q.umf = R(rstate(27));
        return;
    }
    const int krel = q.krel;
    q.thlu = W(W_THLU, krel - 1);
    q.qtu = W(W_QTU, krel - 1);
    q.uu = W(W_UU, krel - 1);
    q.vu = W(W_VU, krel - 1);
    q.thvu = W(W_THVU, krel - 1);
    q.wu = R(out(a.wu, krel - 1));
    q.umf = R(out(a.umf, krel - 1));
}

template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE bool Column<R, D, ZW, FAST>::sort_level(SortState<R, D>& q) const {
    const R rmaxfrac = R(0.10), rbuoy = R(1), rdrag = R(1);
    const R PGFc = R(0.7), criqc = R(0.7e-3);
    const R xlv = R(C.xlv), xls = R(C.xls), cp = R(C.cp), r = R(C.r), g = R(C.g);
    const R rle = R(param(1)), rkm = R(param(2));
    const R dt = R(a.dt);
    constexpr bool kFp32 = sizeof(R) == sizeof(float);
    constexpr double kGuard = kFp32 ? 1.e-5 : 1.e-8;
    auto near = [&](auto dist, auto scale) {   // the branch guard of run_body
        if constexpr (kFp32 || FAST) {
            if (fabs(dist) <= kGuard * fabs(scale)) q.amb = 1;
        }
    };
    D th, qvj, qlj, qij;
    const int k = q.k, krel = q.krel;
    const R pe = q.pe, dpe = q.dpe, exne = q.exne, thle = q.thle, qte = q.qte, ue = q.ue, ve = q.ve;
    const D exe = q.exe;
    // Read once for both iter_xc passes: the environment of layer k, which the loop
    // body does not write, and (issued early) that of layer k+1 for the next level.
    const R thlu_km1 = q.thlu, qtu_km1 = q.qtu;
    const R uu_km1 = q.uu, vu_km1 = q.vu, thvu_km1 = q.thvu;
    const R wu_km1 = q.wu;
    const EnvLevelOf<D> ek = env_level_upper(k), en = env_level_lower(k + 1);
    const R z0k = R(ek.z0), dp0k = R(q.dp0), thv0top_k = R(ek.thv0top);
    const R ss_thl = R(ek.ssthl), ss_qt = R(ek.ssqt), ss_u = R(ek.ssu), ss_v = R(ek.ssv);
    const D ps0k = ek.ps0, exns0k = ek.exns0;
    R thlue = thlu_km1;
    R qtue = qtu_km1;
    R wue = wu_km1;
    R wtw = q.wtw, wtwb = q.wtw;
    const R umf_km1 = q.umf;
    R umfk = 0, ferk = 0, fdrk = 0, drage = 0, bogbot = 0, bogtop = 0;
    // Level-k results of an iter_xc pass.  Each pass overwrites the last and none
    // reads them back, so they are stored once, after the passes.
    R reik = 0, thluk = 0, qtuk = 0, uuk = 0, vuk = 0, thvuk = 0, dwtenk = 0, ditenk = 0;
    // the environment at pe does not change between the iter_xc passes
    R thv0j;
    D es, qs;
    if (k == krel) {
        if (T.conden_x(pe, exe, thle, qte, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return false; }
        thv0j = thv_of(th, qvj, qlj, qij);
        T.qsat_es_qs(D(thle * exne), pe, es, qs);
    } else {
        if constexpr (kRec) {
            if (!(ek.thv0mid > 0.0)) { q.exit_code = EX_CONDEN; return false; }
            thv0j = R(ek.thv0mid);
            qs = ek.qs0mid;
        } else {
            D tv;
            if (!env_mid(k, tv, qs)) { q.exit_code = EX_CONDEN; return false; }
            thv0j = R(tv);
        }
    }
    const R rho0j = pe / (r * thv0j * exne);
    const R excess0 = qte - R(qs);
    for (int iter_xc = 1; iter_xc <= 2; ++iter_xc) {
        wtw = wu_km1 * wu_km1;
        if (T.conden_x(pe, exe, thlue, qtue, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return false; }
        near(qlj + qij - criqc, criqc);
        if ((R(qlj) + R(qij)) > criqc) {
            const R qlr = R(qlj), qir = R(qij);
            const R exql = ((qlr + qir) - criqc) * qlr / (qlr + qir);
            const R exqi = ((qlr + qir) - criqc) * qir / (qlr + qir);
            qtue = qtue - exql - exqi;
            thlue = thlue + (xlv / cp / exne) * exql + (xls / cp / exne) * exqi;
            // unchanged arguments give unchanged results, so only re-adjust here
            if (T.conden_x(pe, exe, thlue, qtue, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return false; }
        }
        const R thvj = thv_of(th, qvj, qlj, qij);
        T.qsat_es_qs(D(thlue * exne), pe, es, qs);
        const R excessu = qtue - R(qs);
        near(excessu, qtue);
        near(excess0, qte);
        const R cridis = rle * q.scaleh;
        R xc;
        if ((excessu <= R(0) && excess0 <= R(0)) || (excessu >= R(0) && excess0 >= R(0))) {
            xc = fmin(R(1), fmax(R(0), R(1) - R(2) * rbuoy * g * cridis / (wue * wue) * (R(1) - thvj / thv0j)));
        } else {
            const R xsat = excessu / (excessu - excess0);
            const R thlxsat = thlue + xsat * (thle - thlue);
            const R qtxsat = qtue + xsat * (qte - qtue);
            if (T.conden_x(pe, exe, thlxsat, qtxsat, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return false; }
            const R thvxsat = thv_of(th, qvj, qlj, qij);
            R x_cu = 0, x_en = 0;
            for (int kk = 1; kk <= 2; ++kk) {
                R thv_x0, thv_x1;
                if (kk == 1) {
                    thv_x0 = thvj;
                    thv_x1 = (R(1) - R(1) / xsat) * thvj + (R(1) / xsat) * thvxsat;
                } else {
                    thv_x1 = thv0j;
                    thv_x0 = (xsat / (xsat - R(1))) * thv0j + (R(1) / (R(1) - xsat)) * thvxsat;
                }
                const R aquad = wue * wue;
                const R bquad = R(2) * rbuoy * g * cridis * (thv_x1 - thv_x0) / thv0j - R(2) * (wue * wue);
                const R cquad = R(2) * rbuoy * g * cridis * (thv_x0 - thv0j) / thv0j + (wue * wue);
                R xs1 = 0, xs2 = 0;
                int status;
                near(bquad * bquad - R(4) * aquad * cquad, bquad * bquad + fabs(R(4) * aquad * cquad));
                if (kk == 1) {
                    if ((bquad * bquad - R(4) * aquad * cquad) >= R(0)) {
                        roots(aquad, bquad, cquad, xs1, xs2, status);
                        near(xsat - fmin(xs1, xs2), R(1));
                        x_cu = fmin(R(1), fmax(R(0), fmin(xsat, fmin(xs1, xs2))));
                    } else {
                        x_cu = xsat;
                    }
                } else {
                    if ((bquad * bquad - R(4) * aquad * cquad) >= R(0)) {
                        roots(aquad, bquad, cquad, xs1, xs2, status);
                        x_en = fmin(R(1), fmax(R(0), fmax(xsat, fmin(xs1, xs2))));
                    } else {
                        x_en = R(1);
                    }
                }
            }
            xc = (x_cu == xsat) ? fmax(x_cu, x_en) : x_cu;
        }
        near(xc - R(0.5), R(1));
        const R ee2 = xc * xc;
        const R ud2 = R(1) - R(2) * xc + xc * xc;
        reik = (R(0.5) * rkm / z0k / g / rho0j);
        if (xc > R(0.5))
            reik = fmin(reik, R(0.9) * ulog(dp0k / g / dt / umf_km1 + R(1)) / dpe / (R(2) * xc - R(1)));
        ferk = reik * ee2;
        fdrk = reik * ud2;
        if constexpr (ZW) {
            if (a.zw.ent) {
                // zwshcu.F90:2818-2844: entrainment from the updraft buoyancy
                const R bog = rbuoy * (thvu_km1 / q.thvebot - R(1)) * g;
                ferk = R(a.zw.ent0) * bog / fmax(wue * wue, R(1.0e-4));
                const R fer_min = bog > R(1.e-4) ? R(1.e-4) : R(0);
                ferk = fmin(fmax(ferk, fer_min), R(3.0e-2));
            }
        }
        umfk = umf_km1 * uexp(dpe * (ferk - fdrk));
        if (ferk * dpe < R(1.e-4)) {
            thluk = thlu_km1 + (thle + ss_thl * dpe / R(2) - thlu_km1) * ferk * dpe;
            qtuk = qtu_km1 + (qte + ss_qt * dpe / R(2) - qtu_km1) * ferk * dpe;
            uuk = uu_km1 + (ue + ss_u * dpe / R(2) - uu_km1) * ferk * dpe - PGFc * ss_u * dpe;
            vuk = vu_km1 + (ve + ss_v * dpe / R(2) - vu_km1) * ferk * dpe - PGFc * ss_v * dpe;
        } else {
            const R ef = uexp(-ferk * dpe);
            thluk = (thle + ss_thl / ferk - ss_thl * dpe / R(2)) -
                    (thle + ss_thl * dpe / R(2) - thlu_km1 + ss_thl / ferk) * ef;
            qtuk = (qte + ss_qt / ferk - ss_qt * dpe / R(2)) -
                   (qte + ss_qt * dpe / R(2) - qtu_km1 + ss_qt / ferk) * ef;
            uuk = (ue + (R(1) - PGFc) * ss_u / ferk - ss_u * dpe / R(2)) -
                  (ue + ss_u * dpe / R(2) - uu_km1 + (R(1) - PGFc) * ss_u / ferk) * ef;
            vuk = (ve + (R(1) - PGFc) * ss_v / ferk - ss_v * dpe / R(2)) -
                  (ve + ss_v * dpe / R(2) - vu_km1 + (R(1) - PGFc) * ss_v / ferk) * ef;
        }
        if (T.conden_x(ps0k, exns0k, thluk, qtuk, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return false; }
        near(qlj + qij - criqc, criqc);
        if ((R(qlj) + R(qij)) > criqc) {
            const R qlr = R(qlj), qir = R(qij);
            const R exql = ((qlr + qir) - criqc) * qlr / (qlr + qir);
            const R exqi = ((qlr + qir) - criqc) * qir / (qlr + qir);
            qtuk = qtuk - exql - exqi;
            thluk = thluk + (xlv / cp / R(exns0k)) * exql + (xls / cp / R(exns0k)) * exqi;
            dwtenk = exql;
            ditenk = exqi;
            if (T.conden_x(ps0k, exns0k, thluk, qtuk, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return false; }
        } else {
            dwtenk = R(0);
            ditenk = R(0);
        }
        thvuk = thv_of(th, qvj, qlj, qij);
        bogbot = rbuoy * (thvu_km1 / q.thvebot - R(1));
        bogtop = rbuoy * (thvuk / thv0top_k - R(1));
        const R delbog = bogtop - bogbot;
        drage = ferk * (R(1) + rdrag);
        const R expfac = uexp(R(-2) * drage * dpe);
        wtwb = wtw;
        if (drage * dpe > R(1.e-3))
            wtw = wtw * expfac + (delbog + (R(1) - expfac) * (bogbot + delbog / (R(-2) * drage * dpe))) / (rho0j * drage);
        else
            wtw = wtw + dpe * (bogbot + bogtop) / rho0j;
        near(wtw, wtwb);
        near(bogtop, R(1));
        if (wtw > R(0)) {
            thlue = R(0.5) * (thlu_km1 + thluk);
            qtue = R(0.5) * (qtu_km1 + qtuk);
            wue = R(0.5) * sqrt(fmax(wtwb + wtw, R(0)));
        } else {
            break;   // go to 111
        }
    }
    // 111 continue
    // Updraft tracers (uwshcu.F90:2592-2614).  Nothing in an iter_xc pass reads
    // them and each pass overwrites the last, so they are formed once, from the
    // fer(k) of the pass that ended the loop.
    if (ncnst < kTrLimited) {
    } else if (ferk * dpe < R(1.e-4)) {
        for (int m = kTrLimited; m <= ncnst; ++m) {
            if (!tr_moved(m)) continue;
            const R tre = q.tr_mid ? R(trin(m, q.ktr)) : R(trin(m, q.ktr)) + WT(0, m, q.ktr) * q.pe_tr;
            WT(1, m, k) = WT(1, m, k - 1) + (tre + WT(0, m, k) * dpe / R(2) - WT(1, m, k - 1)) * ferk * dpe;
        }
    } else {
        const R ef = uexp(-ferk * dpe);
        for (int m = kTrLimited; m <= ncnst; ++m) {
            if (!tr_moved(m)) continue;
            const R tre = q.tr_mid ? R(trin(m, q.ktr)) : R(trin(m, q.ktr)) + WT(0, m, q.ktr) * q.pe_tr;
            const R sst = WT(0, m, k);
            WT(1, m, k) = (tre + sst / ferk - sst * dpe / R(2)) -
                          (tre + sst * dpe / R(2) - WT(1, m, k - 1) + sst / ferk) * ef;
        }
    }
    q.rho0j = rho0j;
    q.drage = drage;
    q.bogbot = bogbot;
    q.bogtop = bogtop;
    q.wtwb = wtwb;
    q.fer = ferk;
    if (k == krel) q.fer_krel = ferk;
    if (umfk == R(0)) wtw = R(-1);
    if (bogtop > R(0) && wtw > R(0)) q.kbup = k;
    const bool top = wtw <= R(0);   // go to 45
    if (!top) {
        const R wuk = sqrt(wtw);
        if constexpr (kRec) P(P_WU, k) = wuk;
        else out(a.wu, k) = D(wuk);
        q.kwu = q.kwu > k ? q.kwu : k;
        if (wuk > R(100)) { q.exit_code = EX_WU; return false; }
        const R rhos0j = R(ps0k) / (r * R(0.5) * (R(en.thv0bot) + thv0top_k) * R(exns0k));
        R ufrck = umfk / (rhos0j * wuk);
        near(ufrck - rmaxfrac, rmaxfrac);
        if (ufrck > rmaxfrac) {
            q.limit_ufrc = 1;
            ufrck = rmaxfrac;
            umfk = rmaxfrac * rhos0j * wuk;
            fdrk = ferk - ulog(umfk / umf_km1) / dpe;
        }
        if (q.iter == 3) P(W_UFRC, k) = ufrck;
        q.wu = R(D(wuk));
        q.umf = R(D(umfk));
    }
    // The stages that follow read the levels up to the last iteration's cloud top: the first
    // two keep only wu, whose values above the cloud top are an output.
    if (q.iter == 3) {
        P(W_REI, k) = reik;
        P(W_FDR, k) = fdrk;
        P(W_DWTEN, k) = dwtenk;
        P(W_DITEN, k) = ditenk;
        P(W_THLU, k) = thluk;
        P(W_QTU, k) = qtuk;
        P(W_UU, k) = uuk;
        P(W_VU, k) = vuk;
        if constexpr (kRec) {
            P(P_UMF, k) = umfk;
        } else {
            out(a.umf, k) = D(umfk);
        }
    }
    if (top) {
        q.kpen = k;
        return false;
    }
    if (k == mkx - 1) {
        // the updraft reaches the last level: the cloud top stays at the release level, whose
        // plume the cloud-top stage reads
        q.fer = q.fer_krel;
        sort_release(q);
        return false;
    }
    q.thlu = thluk;
    q.qtu = qtuk;
    q.uu = uuk;
    q.vu = vuk;
    q.thvu = thvuk;
    q.wtw = wtw;
    q.pe = R(en.p0);
    q.dpe = R(en.dp0);
    q.dp0 = en.dp0;
    q.exne = R(en.exn0);
    if constexpr (sizeof(R) == sizeof(double)) q.exe = en.exn0;   // = exnf(pe), pe = p0(k+1)
    else q.exe = T.exnf(D(q.pe));
    q.thvebot = R(en.thv0bot);
    q.thle = R(en.thl0);
    q.qte = R(en.qt0);
    q.ue = R(en.u0);
    q.ve = R(en.v0);
    q.ktr = k + 1;
    q.tr_mid = true;
    q.k = k + 1;
    return true;
}

// 45 continue: the cloud top.  q.thlu, q.qtu and q.wu are those of interface kpen-1 and
// q.fer is fer(kpen).
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE void Column<R, D, ZW, FAST>::sort_top(SortState<R, D>& q) const {
    const R criqc = R(0.7e-3), xlv = R(C.xlv), xls = R(C.xls), cp = R(C.cp), r = R(C.r), g = R(C.g);
    constexpr bool kFp32 = sizeof(R) == sizeof(float);
    constexpr double kGuard = kFp32 ? 1.e-5 : 1.e-8;
    auto near = [&](auto dist, auto scale) {
        if constexpr (kFp32 || FAST) {
            if (fabs(dist) <= kGuard * fabs(scale)) q.amb = 1;
        }
    };
    D th, qvj, qlj, qij;
    const int kpen = q.kpen;
    const EnvLevelOf<D> e = env_level(kpen), eb = env_level(kpen - 1);
    R ppen;
    if (q.drage == R(0)) {
        const R aquad = (q.bogtop - q.bogbot) / R(e.ps0 - eb.ps0);
        const R bquad = R(2) * q.bogbot;
        const R cquad = -(q.wu * q.wu) * q.rho0j;
        R xc1 = 0, xc2 = 0;
        int status;
        roots(aquad, bquad, cquad, xc1, xc2, status);
        const R dpk = R(e.dp0);
        if (status == 0) {
            if (xc1 <= R(0) && xc2 <= R(0)) {
                ppen = fmax(xc1, xc2);
                ppen = fmin(R(0), fmax(-dpk, ppen));
            } else if (xc1 > R(0) && xc2 > R(0)) {
                ppen = -dpk;
            } else {
                ppen = fmin(xc1, xc2);
                ppen = fmin(R(0), fmax(-dpk, ppen));
            }
        } else {
            ppen = -dpk;
        }
    } else {
        ppen = compute_ppen(q.wtwb, q.drage, q.bogbot, q.bogtop, q.rho0j, R(e.dp0));
    }
    q.ppen = ppen;
    if (ppen == -R(e.dp0) || ppen == R(0)) q.limit_ppen = 1;
    R thlu_top, qtu_top;
    {
        const R ferp = q.fer, thl0p = R(e.thl0), ssthlp = R(e.ssthl);
        const R qt0p = R(e.qt0), ssqtp = R(e.ssqt);
        if (ferp * (-ppen) < R(1.e-4)) {
            thlu_top = q.thlu + (thl0p + ssthlp * (-ppen) / R(2) - q.thlu) * ferp * (-ppen);
            qtu_top = q.qtu + (qt0p + ssqtp * (-ppen) / R(2) - q.qtu) * ferp * (-ppen);
        } else {
            const R ef = uexp(-ferp * (-ppen));
            thlu_top = (thl0p + ssthlp / ferp - ssthlp * (-ppen) / R(2)) -
                       (thl0p + ssthlp * (-ppen) / R(2) - q.thlu + ssthlp / ferp) * ef;
            qtu_top = (qt0p + ssqtp / ferp - ssqtp * (-ppen) / R(2)) -
                      (qt0p + ssqtp * (-ppen) / R(2) - q.qtu + ssqtp / ferp) * ef;
        }
    }
    const R ptop = R(eb.ps0) + ppen;
    if (T.conden(ptop, thlu_top, qtu_top, th, qvj, qlj, qij)) { q.exit_code = EX_CONDEN; return; }
    near(qlj + qij - criqc, criqc);
    const R exntop = R(upow(D(ptop) / C.p00, C.rovcp));
    R dw = R(0), di = R(0);
    if ((R(qlj) + R(qij)) > criqc) {
        const R qlr = R(qlj), qir = R(qij);
        dw = ((qlr + qir) - criqc) * qlr / (qlr + qir);
        di = ((qlr + qir) - criqc) * qir / (qlr + qir);
        qtu_top = qtu_top - dw - di;
        thlu_top = thlu_top + (xlv / cp / exntop) * dw + (xls / cp / exntop) * di;
    }
    if (q.iter == 3) {
        P(W_DWTEN, kpen) = dw;
        P(W_DITEN, kpen) = di;
    }
    q.thlu_top = thlu_top;
    q.qtu_top = qtu_top;
    const R rhos0j = R(eb.ps0) / (r * R(0.5) * (R(e.thv0bot) + R(eb.thv0top)) * R(eb.exns0));
    q.cush = D(R(in(a.zs0, kpen - 1)) - ppen / rhos0j / g);
}

// A listed column's scalars: those of its closure at the start, what S11 set at its end
// (the other saved scalars still hold the closure's values).
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE void Column<R, D, ZW, FAST>::sort_load(SortState<R, D>& q) const {
    q.cush = rstate(0);
    q.prel = R(rstate(13));
    q.thv0rel = R(rstate(14));
    q.wlcl = R(rstate(16));
    q.krel = (int)rstate(33);
    q.limit_ufrc = (int)rstate(36);
    q.limit_ppen = (int)rstate(37);
    q.amb = (int)rstate(39);
    q.exit_code = EX_NONE;
    q.kwu = 0;
}
template <class R, class D, bool ZW, bool FAST>
UWSHCU_HD UW_INLINE void Column<R, D, ZW, FAST>::sort_store(const SortState<R, D>& q, bool second_pass) const {
    rstate(34) = (double)q.kbup;
    rstate(35) = (double)q.kpen;
    rstate(36) = (double)q.limit_ufrc;
    rstate(37) = (double)q.limit_ppen;
    rstate(39) = (double)q.amb;
    if (q.exit_code != EX_NONE) {
        write_exit();
        write_diag(0, q.exit_code, second_pass ? 2 : 1, q.amb);
        rstate(RS_CONT) = 0.0;
        return;
    }
    rstate(29) = (double)q.kwu;
    rstate(0) = (double)val(q.cush);
    rstate(18) = (double)val(q.ppen);
    rstate(19) = (double)val(q.thlu_top);
    rstate(20) = (double)val(q.qtu_top);
    rstate(RS_CONT) = 1.0;
}

}  // namespace uwshcu
#endif
