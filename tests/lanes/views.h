// Smem views of a group, each array (those the kernel addresses as one together) in a region of its
// own. Included by react_kernel.h in front of the views of the device.
template <int N, int R, int G>
double* setup_views(Smem<N, R>& S, unsigned char*, const BlobLayout& BL, int, double*) {
  constexpr int n = N + 1;
  static emu::Region ctl, arr, perm, lu, lp, js, rec;
  S.sp = (const SpRec*)emu_blob(BL.off_sp, BL.off_rx);
  S.rx = (const RxRec*)emu_blob(BL.off_rx, BL.off_effsp);
  S.effsp = (const int*)emu_blob(BL.off_effsp, BL.off_effval);
  S.effval = (const double*)emu_blob(BL.off_effval, BL.off_incq);
  S.incq = (const int*)emu_blob(BL.off_incq, BL.off_incnu);
  S.incnu = (const double*)emu_blob(BL.off_incnu, BL.off_kblk);
  S.kblk = (const int*)emu_blob(BL.off_kblk, BL.off_blk);
  S.blk = (const int*)emu_blob(BL.off_blk, BL.bytes);
  S.sC = emu::region<double>(arr, 5 * N + R);
  S.sG = S.sC + N;
  S.sH = S.sG + N;
  S.sHm = S.sH + N;
  S.sCpm = S.sHm + N;
  S.q = S.sCpm + N;
  S.perm = emu::region<int>(perm, n);
  S.LU = emu::region<double>(lu, n * n);
  S.Lp = (Cell<N, R, G>::lu_global && G == 32) ? emu::region<double>(lp, n) : nullptr;
  S.Js = emu::region<double>(js, n * n);
  S.jrec = emu::region<double>(rec, 5 * R);
  return emu::region<double>(ctl, CTL_DOUBLES, true);
}
