! Generated by gen_bindings.py from include/imsrg_hip.h: bind(C) interfaces
! of libimsrg_hip.so for a Fortran host (iso_c_binding, Fortran 2003).
module imsrg_hip_c
  use, intrinsic :: iso_c_binding
  implicit none
  interface
    function imsrg_last_error() bind(C, name="imsrg_last_error")
      import
      type(c_ptr) :: imsrg_last_error
    end function imsrg_last_error
    function imsrg_basis_create(norb, n, l, jj2, tz2, hole, out) bind(C, name="imsrg_basis_create")
      import
      integer(c_int) :: imsrg_basis_create
      integer(c_int), value :: norb
      integer(c_int), dimension(*) :: n
      integer(c_int), dimension(*) :: l
      integer(c_int), dimension(*) :: jj2
      integer(c_int), dimension(*) :: tz2
      integer(c_int), dimension(*) :: hole
      type(c_ptr), intent(out) :: out
    end function imsrg_basis_create
    function imsrg_basis_destroy(b) bind(C, name="imsrg_basis_destroy")
      import
      integer(c_int) :: imsrg_basis_destroy
      type(c_ptr), value :: b
    end function imsrg_basis_destroy
    function imsrg_basis_size(b, what) bind(C, name="imsrg_basis_size")
      import
      integer(c_int64_t) :: imsrg_basis_size
      type(c_ptr), value :: b
      integer(c_int), value :: what
    end function imsrg_basis_size
    function imsrg_basis_channels(b, dims, goff, jtp) bind(C, name="imsrg_basis_channels")
      import
      integer(c_int) :: imsrg_basis_channels
      type(c_ptr), value :: b
      integer(c_int), dimension(*) :: dims
      integer(c_int64_t), dimension(*) :: goff
      integer(c_int), dimension(*) :: jtp
    end function imsrg_basis_channels
    function imsrg_basis_pairs(b, q, cls, out) bind(C, name="imsrg_basis_pairs")
      import
      integer(c_int) :: imsrg_basis_pairs
      type(c_ptr), value :: b
      integer(c_int), value :: q
      integer(c_int), value :: cls
      integer(c_int), dimension(*) :: out
    end function imsrg_basis_pairs
    function imsrg_basis_cc(b, rlen, ncol, ccoff, wcoff, jtp) bind(C, name="imsrg_basis_cc")
      import
      integer(c_int) :: imsrg_basis_cc
      type(c_ptr), value :: b
      integer(c_int), dimension(*) :: rlen
      integer(c_int), dimension(*) :: ncol
      integer(c_int64_t), dimension(*) :: ccoff
      integer(c_int64_t), dimension(*) :: wcoff
      integer(c_int), dimension(*) :: jtp
    end function imsrg_basis_cc
    function imsrg_basis_sixj(b, j1, j2, j3, j4, j5, j6) bind(C, name="imsrg_basis_sixj")
      import
      real(c_double) :: imsrg_basis_sixj
      type(c_ptr), value :: b
      integer(c_int), value :: j1
      integer(c_int), value :: j2
      integer(c_int), value :: j3
      integer(c_int), value :: j4
      integer(c_int), value :: j5
      integer(c_int), value :: j6
    end function imsrg_basis_sixj
    function imsrg_set_path(b, path) bind(C, name="imsrg_set_path")
      import
      integer(c_int) :: imsrg_set_path
      type(c_ptr), value :: b
      integer(c_int), value :: path
    end function imsrg_set_path
    function imsrg_alloc(count, out) bind(C, name="imsrg_alloc")
      import
      integer(c_int) :: imsrg_alloc
      integer(c_int64_t), value :: count
      type(c_ptr), intent(out) :: out
    end function imsrg_alloc
    function imsrg_free(p) bind(C, name="imsrg_free")
      import
      integer(c_int) :: imsrg_free
      type(c_ptr), value :: p
    end function imsrg_free
    function imsrg_op_put(b, op, q, g, host) bind(C, name="imsrg_op_put")
      import
      integer(c_int) :: imsrg_op_put
      type(c_ptr), value :: b
      type(c_ptr), value :: op
      integer(c_int), value :: q
      integer(c_int), value :: g
      real(c_double), dimension(*) :: host
    end function imsrg_op_put
    function imsrg_op_get(b, op, q, g, host) bind(C, name="imsrg_op_get")
      import
      integer(c_int) :: imsrg_op_get
      type(c_ptr), value :: b
      type(c_ptr), value :: op
      integer(c_int), value :: q
      integer(c_int), value :: g
      real(c_double), dimension(*) :: host
    end function imsrg_op_get
    function imsrg_vectorize(b, op, vec, stream) bind(C, name="imsrg_vectorize")
      import
      integer(c_int) :: imsrg_vectorize
      type(c_ptr), value :: b
      type(c_ptr), value :: op
      type(c_ptr), value :: vec
      type(c_ptr), value :: stream
    end function imsrg_vectorize
    function imsrg_repackage(b, vec, herm, op, stream) bind(C, name="imsrg_repackage")
      import
      integer(c_int) :: imsrg_repackage
      type(c_ptr), value :: b
      type(c_ptr), value :: vec
      integer(c_int), value :: herm
      type(c_ptr), value :: op
      type(c_ptr), value :: stream
    end function imsrg_repackage
    function imsrg_write_op_bin(b, op, path, stream) bind(C, name="imsrg_write_op_bin")
      import
      integer(c_int) :: imsrg_write_op_bin
      type(c_ptr), value :: b
      type(c_ptr), value :: op
      character(kind=c_char), dimension(*) :: path
      type(c_ptr), value :: stream
    end function imsrg_write_op_bin
    function imsrg_read_op_bin(b, path, herm, op, stream) bind(C, name="imsrg_read_op_bin")
      import
      integer(c_int) :: imsrg_read_op_bin
      type(c_ptr), value :: b
      character(kind=c_char), dimension(*) :: path
      integer(c_int), value :: herm
      type(c_ptr), value :: op
      type(c_ptr), value :: stream
    end function imsrg_read_op_bin
    function imsrg_h0_harm_osc(b, hw, htype, lawson_beta, com_hw, mass, h, stream) bind(C, name="imsrg_h0_harm_osc")
      import
      integer(c_int) :: imsrg_h0_harm_osc
      type(c_ptr), value :: b
      real(c_double), value :: hw
      integer(c_int), value :: htype
      real(c_double), value :: lawson_beta
      real(c_double), value :: com_hw
      integer(c_int), value :: mass
      type(c_ptr), value :: h
      type(c_ptr), value :: stream
    end function imsrg_h0_harm_osc
    function imsrg_read_me2j( &
        b, path, nfile, n, l, jj, tz, hw, htype, lawson_beta, com_hw, mass, h, stream) &
        bind(C, name="imsrg_read_me2j")
      import
      integer(c_int) :: imsrg_read_me2j
      type(c_ptr), value :: b
      character(kind=c_char), dimension(*) :: path
      integer(c_int), value :: nfile
      integer(c_int), dimension(*) :: n
      integer(c_int), dimension(*) :: l
      integer(c_int), dimension(*) :: jj
      integer(c_int), dimension(*) :: tz
      real(c_double), value :: hw
      integer(c_int), value :: htype
      real(c_double), value :: lawson_beta
      real(c_double), value :: com_hw
      integer(c_int), value :: mass
      type(c_ptr), value :: h
      type(c_ptr), value :: stream
    end function imsrg_read_me2j
    function imsrg_hartree_fock(b, h, maxit, ehf, iterations, coefs, stream) bind(C, name="imsrg_hartree_fock")
      import
      integer(c_int) :: imsrg_hartree_fock
      type(c_ptr), value :: b
      type(c_ptr), value :: h
      integer(c_int), value :: maxit
      type(c_ptr), value :: ehf
      integer(c_int), dimension(*) :: iterations
      type(c_ptr), value :: coefs
      type(c_ptr), value :: stream
    end function imsrg_hartree_fock
    function imsrg_sqop_to_hf(b, coefs, op, herm, stream) bind(C, name="imsrg_sqop_to_hf")
      import
      integer(c_int) :: imsrg_sqop_to_hf
      type(c_ptr), value :: b
      type(c_ptr), value :: coefs
      type(c_ptr), value :: op
      integer(c_int), value :: herm
      type(c_ptr), value :: stream
    end function imsrg_sqop_to_hf
    function imsrg_commutator_110(b, l, lherm, r, rherm, value, stream) bind(C, name="imsrg_commutator_110")
      import
      integer(c_int) :: imsrg_commutator_110
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      real(c_double), dimension(*) :: value
      type(c_ptr), value :: stream
    end function imsrg_commutator_110
    function imsrg_commutator_220(b, l, lherm, r, rherm, value, stream) bind(C, name="imsrg_commutator_220")
      import
      integer(c_int) :: imsrg_commutator_220
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      real(c_double), dimension(*) :: value
      type(c_ptr), value :: stream
    end function imsrg_commutator_220
    function imsrg_commutator_e0(b, l, lherm, r, rherm, res, stream) bind(C, name="imsrg_commutator_e0")
      import
      integer(c_int) :: imsrg_commutator_e0
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      type(c_ptr), value :: stream
    end function imsrg_commutator_e0
    function imsrg_commutator_111(b, l, lherm, r, rherm, res, resherm, stream) bind(C, name="imsrg_commutator_111")
      import
      integer(c_int) :: imsrg_commutator_111
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_commutator_111
    function imsrg_commutator_121(b, l, lherm, r, rherm, res, resherm, stream) bind(C, name="imsrg_commutator_121")
      import
      integer(c_int) :: imsrg_commutator_121
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_commutator_121
    function imsrg_commutator_122(b, l, lherm, r, rherm, res, resherm, stream) bind(C, name="imsrg_commutator_122")
      import
      integer(c_int) :: imsrg_commutator_122
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_commutator_122
    function imsrg_commutator_222_pp_hh( &
        b, l, lherm, r, rherm, res, resherm, w1, w2, stream) &
        bind(C, name="imsrg_commutator_222_pp_hh")
      import
      integer(c_int) :: imsrg_commutator_222_pp_hh
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: w1
      type(c_ptr), value :: w2
      type(c_ptr), value :: stream
    end function imsrg_commutator_222_pp_hh
    function imsrg_commutator_221( &
        b, l, lherm, r, rherm, res, resherm, w1, w2, stream) &
        bind(C, name="imsrg_commutator_221")
      import
      integer(c_int) :: imsrg_commutator_221
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: w1
      type(c_ptr), value :: w2
      type(c_ptr), value :: stream
    end function imsrg_commutator_221
    function imsrg_calculate_cross_coupled(b, op, herm, cc, stream) bind(C, name="imsrg_calculate_cross_coupled")
      import
      integer(c_int) :: imsrg_calculate_cross_coupled
      type(c_ptr), value :: b
      type(c_ptr), value :: op
      integer(c_int), value :: herm
      type(c_ptr), value :: cc
      type(c_ptr), value :: stream
    end function imsrg_calculate_cross_coupled
    function imsrg_commutator_222_ph( &
        b, lcc, lherm, rcc, rherm, res, resherm, wcc, stream) &
        bind(C, name="imsrg_commutator_222_ph")
      import
      integer(c_int) :: imsrg_commutator_222_ph
      type(c_ptr), value :: b
      type(c_ptr), value :: lcc
      integer(c_int), value :: lherm
      type(c_ptr), value :: rcc
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: wcc
      type(c_ptr), value :: stream
    end function imsrg_commutator_222_ph
    function imsrg_commutator_222_ph_noalloc( &
        b, lcc, lherm, rcc, rherm, res, resherm, stream) &
        bind(C, name="imsrg_commutator_222_ph_noalloc")
      import
      integer(c_int) :: imsrg_commutator_222_ph_noalloc
      type(c_ptr), value :: b
      type(c_ptr), value :: lcc
      integer(c_int), value :: lherm
      type(c_ptr), value :: rcc
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_commutator_222_ph_noalloc
    function imsrg_add_sq_op(b, a, ax, b_, bx, c, stream) bind(C, name="imsrg_add_sq_op")
      import
      integer(c_int) :: imsrg_add_sq_op
      type(c_ptr), value :: b
      type(c_ptr), value :: a
      real(c_double), value :: ax
      type(c_ptr), value :: b_
      real(c_double), value :: bx
      type(c_ptr), value :: c
      type(c_ptr), value :: stream
    end function imsrg_add_sq_op
    function imsrg_mat_frob_norm(b, op, value, stream) bind(C, name="imsrg_mat_frob_norm")
      import
      integer(c_int) :: imsrg_mat_frob_norm
      type(c_ptr), value :: b
      type(c_ptr), value :: op
      real(c_double), dimension(*) :: value
      type(c_ptr), value :: stream
    end function imsrg_mat_frob_norm
    function imsrg_build_gs_white(b, h, eta, stream) bind(C, name="imsrg_build_gs_white")
      import
      integer(c_int) :: imsrg_build_gs_white
      type(c_ptr), value :: b
      type(c_ptr), value :: h
      type(c_ptr), value :: eta
      type(c_ptr), value :: stream
    end function imsrg_build_gs_white
    function imsrg_build_gs_atan(b, h, eta, stream) bind(C, name="imsrg_build_gs_atan")
      import
      integer(c_int) :: imsrg_build_gs_atan
      type(c_ptr), value :: b
      type(c_ptr), value :: h
      type(c_ptr), value :: eta
      type(c_ptr), value :: stream
    end function imsrg_build_gs_atan
    function imsrg_build_gs_atanxx(b, hold, h, eta, stream) bind(C, name="imsrg_build_gs_atanxx")
      import
      integer(c_int) :: imsrg_build_gs_atanxx
      type(c_ptr), value :: b
      type(c_ptr), value :: hold
      type(c_ptr), value :: h
      type(c_ptr), value :: eta
      type(c_ptr), value :: stream
    end function imsrg_build_gs_atanxx
    function imsrg_mbpt2(b, h, value, stream) bind(C, name="imsrg_mbpt2")
      import
      integer(c_int) :: imsrg_mbpt2
      type(c_ptr), value :: b
      type(c_ptr), value :: h
      real(c_double), dimension(*) :: value
      type(c_ptr), value :: stream
    end function imsrg_mbpt2
    function imsrg_normal_order(b, h, stream) bind(C, name="imsrg_normal_order")
      import
      integer(c_int) :: imsrg_normal_order
      type(c_ptr), value :: b
      type(c_ptr), value :: h
      type(c_ptr), value :: stream
    end function imsrg_normal_order
    function imsrg_flow_create(b, out) bind(C, name="imsrg_flow_create")
      import
      integer(c_int) :: imsrg_flow_create
      type(c_ptr), value :: b
      type(c_ptr), intent(out) :: out
    end function imsrg_flow_create
    function imsrg_flow_destroy(f) bind(C, name="imsrg_flow_destroy")
      import
      integer(c_int) :: imsrg_flow_destroy
      type(c_ptr), value :: f
    end function imsrg_flow_destroy
    function imsrg_flow_set_graphs(f, on) bind(C, name="imsrg_flow_set_graphs")
      import
      integer(c_int) :: imsrg_flow_set_graphs
      type(c_ptr), value :: f
      integer(c_int), value :: on
    end function imsrg_flow_set_graphs
    function imsrg_flow_set_generator(f, generator) bind(C, name="imsrg_flow_set_generator")
      import
      integer(c_int) :: imsrg_flow_set_generator
      type(c_ptr), value :: f
      integer(c_int), value :: generator
    end function imsrg_flow_set_generator
    function imsrg_build_gs_w2(f, h, eta, stream) bind(C, name="imsrg_build_gs_w2")
      import
      integer(c_int) :: imsrg_build_gs_w2
      type(c_ptr), value :: f
      type(c_ptr), value :: h
      type(c_ptr), value :: eta
      type(c_ptr), value :: stream
    end function imsrg_build_gs_w2
    function imsrg_bch_expand( &
        f, hs, g, gherm, h, hherm, conv, maxit, nterms, advals, stream) &
        bind(C, name="imsrg_bch_expand")
      import
      integer(c_int) :: imsrg_bch_expand
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: g
      integer(c_int), value :: gherm
      type(c_ptr), value :: h
      integer(c_int), value :: hherm
      real(c_double), value :: conv
      integer(c_int), value :: maxit
      integer(c_int), dimension(*) :: nterms
      real(c_double), dimension(*) :: advals
      type(c_ptr), value :: stream
    end function imsrg_bch_expand
    function imsrg_transform_sq_op_bch( &
        f, op, opherm, g, conv, maxit, nterms, stream) &
        bind(C, name="imsrg_transform_sq_op_bch")
      import
      integer(c_int) :: imsrg_transform_sq_op_bch
      type(c_ptr), value :: f
      type(c_ptr), value :: op
      integer(c_int), value :: opherm
      type(c_ptr), value :: g
      real(c_double), value :: conv
      integer(c_int), value :: maxit
      integer(c_int), dimension(*) :: nterms
      type(c_ptr), value :: stream
    end function imsrg_transform_sq_op_bch
    function imsrg_dhds(f, hs, dh, stream) bind(C, name="imsrg_dhds")
      import
      integer(c_int) :: imsrg_dhds
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: dh
      type(c_ptr), value :: stream
    end function imsrg_dhds
    function imsrg_magnus_expand(f, dg, dgherm, g, gherm, conv, ncomm, stream) bind(C, name="imsrg_magnus_expand")
      import
      integer(c_int) :: imsrg_magnus_expand
      type(c_ptr), value :: f
      type(c_ptr), value :: dg
      integer(c_int), value :: dgherm
      type(c_ptr), value :: g
      integer(c_int), value :: gherm
      real(c_double), value :: conv
      integer(c_int), dimension(*) :: ncomm
      type(c_ptr), value :: stream
    end function imsrg_magnus_expand
    function imsrg_euler_step(b, g, dg, ds, stream) bind(C, name="imsrg_euler_step")
      import
      integer(c_int) :: imsrg_euler_step
      type(c_ptr), value :: b
      type(c_ptr), value :: g
      type(c_ptr), value :: dg
      real(c_double), value :: ds
      type(c_ptr), value :: stream
    end function imsrg_euler_step
    function imsrg_magnus_step(f, hs, g, dg, h, ds, bch_conv, mag_conv, out, stream) bind(C, name="imsrg_magnus_step")
      import
      integer(c_int) :: imsrg_magnus_step
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: g
      type(c_ptr), value :: dg
      type(c_ptr), value :: h
      real(c_double), value :: ds
      real(c_double), value :: bch_conv
      real(c_double), value :: mag_conv
      real(c_double), dimension(*) :: out
      type(c_ptr), value :: stream
    end function imsrg_magnus_step
    function imsrg_magnus_decouple( &
        f, hs, g, ds, bch_conv, mag_conv, crit_mode, crit_tol, maxsteps, log, steps, stream) &
        bind(C, name="imsrg_magnus_decouple")
      import
      integer(c_int) :: imsrg_magnus_decouple
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: g
      real(c_double), value :: ds
      real(c_double), value :: bch_conv
      real(c_double), value :: mag_conv
      integer(c_int), value :: crit_mode
      real(c_double), value :: crit_tol
      integer(c_int), value :: maxsteps
      real(c_double), dimension(*) :: log
      integer(c_int), dimension(*) :: steps
      type(c_ptr), value :: stream
    end function imsrg_magnus_decouple
    function imsrg_magnus_decouple_chk( &
        f, hs, g, ds, bch_conv, mag_conv, crit_mode, crit_tol, maxsteps, prefix, chk, log, steps, restart_s, stream) &
        bind(C, name="imsrg_magnus_decouple_chk")
      import
      integer(c_int) :: imsrg_magnus_decouple_chk
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: g
      real(c_double), value :: ds
      real(c_double), value :: bch_conv
      real(c_double), value :: mag_conv
      integer(c_int), value :: crit_mode
      real(c_double), value :: crit_tol
      integer(c_int), value :: maxsteps
      character(kind=c_char), dimension(*) :: prefix
      integer(c_int), value :: chk
      real(c_double), dimension(*) :: log
      integer(c_int), dimension(*) :: steps
      type(c_ptr), value :: restart_s
      type(c_ptr), value :: stream
    end function imsrg_magnus_decouple_chk
    function imsrg_omega_checkpoint_name(prefix, s, out, outlen) bind(C, name="imsrg_omega_checkpoint_name")
      import
      integer(c_int) :: imsrg_omega_checkpoint_name
      character(kind=c_char), dimension(*) :: prefix
      real(c_double), value :: s
      character(kind=c_char), dimension(*) :: out
      integer(c_int), value :: outlen
    end function imsrg_omega_checkpoint_name
    function imsrg_batch_create(b, ninst, out) bind(C, name="imsrg_batch_create")
      import
      integer(c_int) :: imsrg_batch_create
      type(c_ptr), value :: b
      integer(c_int), value :: ninst
      type(c_ptr), intent(out) :: out
    end function imsrg_batch_create
    function imsrg_batch_size(f) bind(C, name="imsrg_batch_size")
      import
      integer(c_int) :: imsrg_batch_size
      type(c_ptr), value :: f
    end function imsrg_batch_size
    function imsrg_batch_commutator(f, l, lh, r, rh, res, stream) bind(C, name="imsrg_batch_commutator")
      import
      integer(c_int) :: imsrg_batch_commutator
      type(c_ptr), value :: f
      type(c_ptr), value :: l
      integer(c_int), value :: lh
      type(c_ptr), value :: r
      integer(c_int), value :: rh
      type(c_ptr), value :: res
      type(c_ptr), value :: stream
    end function imsrg_batch_commutator
    function imsrg_batch_bch_expand(f, hs, g, h, conv, maxit, nterms, stream) bind(C, name="imsrg_batch_bch_expand")
      import
      integer(c_int) :: imsrg_batch_bch_expand
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: g
      type(c_ptr), value :: h
      real(c_double), value :: conv
      integer(c_int), value :: maxit
      integer(c_int), dimension(*) :: nterms
      type(c_ptr), value :: stream
    end function imsrg_batch_bch_expand
    function imsrg_batch_magnus_expand(f, dg, g, conv, ncomm, stream) bind(C, name="imsrg_batch_magnus_expand")
      import
      integer(c_int) :: imsrg_batch_magnus_expand
      type(c_ptr), value :: f
      type(c_ptr), value :: dg
      type(c_ptr), value :: g
      real(c_double), value :: conv
      integer(c_int), dimension(*) :: ncomm
      type(c_ptr), value :: stream
    end function imsrg_batch_magnus_expand
    function imsrg_batch_magnus_decouple( &
        f, hs, g, ds, bch_conv, mag_conv, crit_tol, maxsteps, e0, steps, nsteps_max, stream) &
        bind(C, name="imsrg_batch_magnus_decouple")
      import
      integer(c_int) :: imsrg_batch_magnus_decouple
      type(c_ptr), value :: f
      type(c_ptr), value :: hs
      type(c_ptr), value :: g
      real(c_double), value :: ds
      real(c_double), value :: bch_conv
      real(c_double), value :: mag_conv
      real(c_double), value :: crit_tol
      integer(c_int), value :: maxsteps
      type(c_ptr), value :: e0
      integer(c_int), dimension(*) :: steps
      integer(c_int), dimension(*) :: nsteps_max
      type(c_ptr), value :: stream
    end function imsrg_batch_magnus_decouple
    function imsrg_commutator_vjp( &
        b, l, lherm, r, rherm, resb, resherm, lb, rb, stream) &
        bind(C, name="imsrg_commutator_vjp")
      import
      integer(c_int) :: imsrg_commutator_vjp
      type(c_ptr), value :: b
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: resb
      integer(c_int), value :: resherm
      type(c_ptr), value :: lb
      type(c_ptr), value :: rb
      type(c_ptr), value :: stream
    end function imsrg_commutator_vjp
    function imsrg_bch_vjp(f, g, h, hherm, conv, maxit, hsb, gb, hb, nterms, stream) bind(C, name="imsrg_bch_vjp")
      import
      integer(c_int) :: imsrg_bch_vjp
      type(c_ptr), value :: f
      type(c_ptr), value :: g
      type(c_ptr), value :: h
      integer(c_int), value :: hherm
      real(c_double), value :: conv
      integer(c_int), value :: maxit
      type(c_ptr), value :: hsb
      type(c_ptr), value :: gb
      type(c_ptr), value :: hb
      integer(c_int), dimension(*) :: nterms
      type(c_ptr), value :: stream
    end function imsrg_bch_vjp
    function imsrg_magnus_vjp(f, eta, g, conv, dgb, etab, gb, ncomm, stream) bind(C, name="imsrg_magnus_vjp")
      import
      integer(c_int) :: imsrg_magnus_vjp
      type(c_ptr), value :: f
      type(c_ptr), value :: eta
      type(c_ptr), value :: g
      real(c_double), value :: conv
      type(c_ptr), value :: dgb
      type(c_ptr), value :: etab
      type(c_ptr), value :: gb
      integer(c_int), dimension(*) :: ncomm
      type(c_ptr), value :: stream
    end function imsrg_magnus_vjp
    function imsrg_white_vjp(b, h, etab, hb, stream) bind(C, name="imsrg_white_vjp")
      import
      integer(c_int) :: imsrg_white_vjp
      type(c_ptr), value :: b
      type(c_ptr), value :: h
      type(c_ptr), value :: etab
      type(c_ptr), value :: hb
      type(c_ptr), value :: stream
    end function imsrg_white_vjp
    function imsrg_generator_vjp(f, h, etab, hb, stream) bind(C, name="imsrg_generator_vjp")
      import
      integer(c_int) :: imsrg_generator_vjp
      type(c_ptr), value :: f
      type(c_ptr), value :: h
      type(c_ptr), value :: etab
      type(c_ptr), value :: hb
      type(c_ptr), value :: stream
    end function imsrg_generator_vjp
    function imsrg_normal_order_vjp(b, hb, tb, stream) bind(C, name="imsrg_normal_order_vjp")
      import
      integer(c_int) :: imsrg_normal_order_vjp
      type(c_ptr), value :: b
      type(c_ptr), value :: hb
      type(c_ptr), value :: tb
      type(c_ptr), value :: stream
    end function imsrg_normal_order_vjp
    function imsrg_flow_forward( &
        f, t, ds, bch_conv, mag_conv, crit_tol, maxsteps, ckpt, e0, steps, stream) &
        bind(C, name="imsrg_flow_forward")
      import
      integer(c_int) :: imsrg_flow_forward
      type(c_ptr), value :: f
      type(c_ptr), value :: t
      real(c_double), value :: ds
      real(c_double), value :: bch_conv
      real(c_double), value :: mag_conv
      real(c_double), value :: crit_tol
      integer(c_int), value :: maxsteps
      integer(c_int), value :: ckpt
      type(c_ptr), value :: e0
      integer(c_int), dimension(*) :: steps
      type(c_ptr), value :: stream
    end function imsrg_flow_forward
    function imsrg_flow_backward(f, tb, stream) bind(C, name="imsrg_flow_backward")
      import
      integer(c_int) :: imsrg_flow_backward
      type(c_ptr), value :: f
      type(c_ptr), value :: tb
      type(c_ptr), value :: stream
    end function imsrg_flow_backward
    function imsrg_flow_grad( &
        f, t, ds, bch_conv, mag_conv, crit_tol, maxsteps, ckpt, tb, e0, steps, stream) &
        bind(C, name="imsrg_flow_grad")
      import
      integer(c_int) :: imsrg_flow_grad
      type(c_ptr), value :: f
      type(c_ptr), value :: t
      real(c_double), value :: ds
      real(c_double), value :: bch_conv
      real(c_double), value :: mag_conv
      real(c_double), value :: crit_tol
      integer(c_int), value :: maxsteps
      integer(c_int), value :: ckpt
      type(c_ptr), value :: tb
      type(c_ptr), value :: e0
      integer(c_int), dimension(*) :: steps
      type(c_ptr), value :: stream
    end function imsrg_flow_grad
    function imsrg_set_gemm_tile(b, family, tile) bind(C, name="imsrg_set_gemm_tile")
      import
      integer(c_int) :: imsrg_set_gemm_tile
      type(c_ptr), value :: b
      integer(c_int), value :: family
      integer(c_int), value :: tile
    end function imsrg_set_gemm_tile
    function imsrg_get_gemm_tile(b, family) bind(C, name="imsrg_get_gemm_tile")
      import
      integer(c_int) :: imsrg_get_gemm_tile
      type(c_ptr), value :: b
      integer(c_int), value :: family
    end function imsrg_get_gemm_tile
    function imsrg_set_term_streams(b, on) bind(C, name="imsrg_set_term_streams")
      import
      integer(c_int) :: imsrg_set_term_streams
      type(c_ptr), value :: b
      integer(c_int), value :: on
    end function imsrg_set_term_streams
    function imsrg_profile_kernel( &
        b, which, l, lherm, r, rherm, res, resherm, w1, w2, lcc, rcc, wcc, iters, ms, stream) &
        bind(C, name="imsrg_profile_kernel")
      import
      integer(c_int) :: imsrg_profile_kernel
      type(c_ptr), value :: b
      integer(c_int), value :: which
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: w1
      type(c_ptr), value :: w2
      type(c_ptr), value :: lcc
      type(c_ptr), value :: rcc
      type(c_ptr), value :: wcc
      integer(c_int), value :: iters
      real(c_double), dimension(*) :: ms
      type(c_ptr), value :: stream
    end function imsrg_profile_kernel
    function imsrg_tensor_create(b, rank, dpar, out) bind(C, name="imsrg_tensor_create")
      import
      integer(c_int) :: imsrg_tensor_create
      type(c_ptr), value :: b
      integer(c_int), value :: rank
      integer(c_int), value :: dpar
      type(c_ptr), intent(out) :: out
    end function imsrg_tensor_create
    function imsrg_tensor_destroy(t) bind(C, name="imsrg_tensor_destroy")
      import
      integer(c_int) :: imsrg_tensor_destroy
      type(c_ptr), value :: t
    end function imsrg_tensor_destroy
    function imsrg_tensor_size(t, what) bind(C, name="imsrg_tensor_size")
      import
      integer(c_int64_t) :: imsrg_tensor_size
      type(c_ptr), value :: t
      integer(c_int), value :: what
    end function imsrg_tensor_size
    function imsrg_tensor_set_form(t, form) bind(C, name="imsrg_tensor_set_form")
      import
      integer(c_int) :: imsrg_tensor_set_form
      type(c_ptr), value :: t
      integer(c_int), value :: form
    end function imsrg_tensor_set_form
    function imsrg_tensor_blocks(t, info, dims, goff) bind(C, name="imsrg_tensor_blocks")
      import
      integer(c_int) :: imsrg_tensor_blocks
      type(c_ptr), value :: t
      integer(c_int), dimension(*) :: info
      integer(c_int), dimension(*) :: dims
      integer(c_int64_t), dimension(*) :: goff
    end function imsrg_tensor_blocks
    function imsrg_tensor_op_put(t, op, q, g, host) bind(C, name="imsrg_tensor_op_put")
      import
      integer(c_int) :: imsrg_tensor_op_put
      type(c_ptr), value :: t
      type(c_ptr), value :: op
      integer(c_int), value :: q
      integer(c_int), value :: g
      real(c_double), dimension(*) :: host
    end function imsrg_tensor_op_put
    function imsrg_tensor_op_get(t, op, q, g, host) bind(C, name="imsrg_tensor_op_get")
      import
      integer(c_int) :: imsrg_tensor_op_get
      type(c_ptr), value :: t
      type(c_ptr), value :: op
      integer(c_int), value :: q
      integer(c_int), value :: g
      real(c_double), dimension(*) :: host
    end function imsrg_tensor_op_get
    function imsrg_ts_commutator_111( &
        t, l, lherm, r, rherm, res, resherm, stream) &
        bind(C, name="imsrg_ts_commutator_111")
      import
      integer(c_int) :: imsrg_ts_commutator_111
      type(c_ptr), value :: t
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_111
    function imsrg_ts_commutator_121( &
        t, l, lherm, r, rherm, res, resherm, stream) &
        bind(C, name="imsrg_ts_commutator_121")
      import
      integer(c_int) :: imsrg_ts_commutator_121
      type(c_ptr), value :: t
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_121
    function imsrg_ts_commutator_211( &
        t, lcc, lccherm, r, rherm, res, resherm, stream) &
        bind(C, name="imsrg_ts_commutator_211")
      import
      integer(c_int) :: imsrg_ts_commutator_211
      type(c_ptr), value :: t
      type(c_ptr), value :: lcc
      integer(c_int), value :: lccherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_211
    function imsrg_ts_commutator_122( &
        t, l, lherm, r, rherm, res, resherm, stream) &
        bind(C, name="imsrg_ts_commutator_122")
      import
      integer(c_int) :: imsrg_ts_commutator_122
      type(c_ptr), value :: t
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_122
    function imsrg_ts_commutator_212( &
        t, l, lherm, r, rherm, res, resherm, stream) &
        bind(C, name="imsrg_ts_commutator_212")
      import
      integer(c_int) :: imsrg_ts_commutator_212
      type(c_ptr), value :: t
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_212
    function imsrg_ts_commutator_222_pp_hh( &
        t, l, lherm, r, rherm, res, resherm, w1, w2, stream) &
        bind(C, name="imsrg_ts_commutator_222_pp_hh")
      import
      integer(c_int) :: imsrg_ts_commutator_222_pp_hh
      type(c_ptr), value :: t
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: w1
      type(c_ptr), value :: w2
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_222_pp_hh
    function imsrg_ts_commutator_221(t, w1, w2, pm, res, resherm, stream) bind(C, name="imsrg_ts_commutator_221")
      import
      integer(c_int) :: imsrg_ts_commutator_221
      type(c_ptr), value :: t
      type(c_ptr), value :: w1
      type(c_ptr), value :: w2
      integer(c_int), value :: pm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_221
    function imsrg_calculate_single_pandya(t, r, rherm, rcc, stream) bind(C, name="imsrg_calculate_single_pandya")
      import
      integer(c_int) :: imsrg_calculate_single_pandya
      type(c_ptr), value :: t
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: rcc
      type(c_ptr), value :: stream
    end function imsrg_calculate_single_pandya
    function imsrg_ts_commutator_222_ph( &
        t, lcc, lccherm, rcc, r, rherm, res, resherm, stream) &
        bind(C, name="imsrg_ts_commutator_222_ph")
      import
      integer(c_int) :: imsrg_ts_commutator_222_ph
      type(c_ptr), value :: t
      type(c_ptr), value :: lcc
      integer(c_int), value :: lccherm
      type(c_ptr), value :: rcc
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator_222_ph
    function imsrg_ts_commutator(t, l, lherm, r, rherm, res, resherm, stream) bind(C, name="imsrg_ts_commutator")
      import
      integer(c_int) :: imsrg_ts_commutator
      type(c_ptr), value :: t
      type(c_ptr), value :: l
      integer(c_int), value :: lherm
      type(c_ptr), value :: r
      integer(c_int), value :: rherm
      type(c_ptr), value :: res
      integer(c_int), value :: resherm
      type(c_ptr), value :: stream
    end function imsrg_ts_commutator
    function imsrg_bch_tensor( &
        t, g, gherm, hs, hsherm, conv, iterations, advals, stream) &
        bind(C, name="imsrg_bch_tensor")
      import
      integer(c_int) :: imsrg_bch_tensor
      type(c_ptr), value :: t
      type(c_ptr), value :: g
      integer(c_int), value :: gherm
      type(c_ptr), value :: hs
      integer(c_int), value :: hsherm
      real(c_double), value :: conv
      integer(c_int), dimension(*) :: iterations
      real(c_double), dimension(*) :: advals
      type(c_ptr), value :: stream
    end function imsrg_bch_tensor
    function imsrg_tensor_frob_norm(t, op, value, stream) bind(C, name="imsrg_tensor_frob_norm")
      import
      integer(c_int) :: imsrg_tensor_frob_norm
      type(c_ptr), value :: t
      type(c_ptr), value :: op
      real(c_double), dimension(*) :: value
      type(c_ptr), value :: stream
    end function imsrg_tensor_frob_norm
    function imsrg_tensor_add(t, a, ax, b, bx, c, stream) bind(C, name="imsrg_tensor_add")
      import
      integer(c_int) :: imsrg_tensor_add
      type(c_ptr), value :: t
      type(c_ptr), value :: a
      real(c_double), value :: ax
      type(c_ptr), value :: b
      real(c_double), value :: bx
      type(c_ptr), value :: c
      type(c_ptr), value :: stream
    end function imsrg_tensor_add
  end interface
end module imsrg_hip_c
