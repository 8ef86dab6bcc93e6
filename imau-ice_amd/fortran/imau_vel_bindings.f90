! imau_vel_bindings.f90 -- GENERATED by gen_bindings.py from include/imau_vel.h; do not edit.
!
! ISO_C_BINDING interface to libimauvel.so for a Fortran host (IMAU-ICE's
! ice_velocity_module calls these; see ice_velocity_module_gpu.f90).
MODULE imau_vel_bindings
  USE ISO_C_BINDING
  IMPLICIT NONE

  INTEGER(C_INT32_T), PARAMETER :: IMAU_BC_INFINITE = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_BC_PERIODIC = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_BC_ZERO = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DHI_EXPLICIT = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DHI_NONE = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DHI_SEMIIMPLICIT = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DYN_DIVA = 4
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DYN_NONE = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DYN_SIA = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DYN_SIA_SSA = 3
  INTEGER(C_INT32_T), PARAMETER :: IMAU_DYN_SSA = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_ARG = -2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_CONFIG = -1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_DEVICE = -6
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_DIVERGED = -4
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_NAN = -3
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_NO_DEVICE = -7
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ERR_STALLED = -5
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HBC_FIXED = 4
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HBC_INFINITE = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HBC_NONE = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HBC_PERIODIC = 3
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HBC_ZERO = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HYDRO_DRY = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HYDRO_MARTIN2011 = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_HYDRO_SATURATED = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_IDEAL_ISMIP_HOM_C = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_IDEAL_ISMIP_HOM_D = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_IDEAL_ISMIP_HOM_E = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_IDEAL_ISMIP_HOM_F = 3
  INTEGER(C_INT32_T), PARAMETER :: IMAU_MARGIN_BC = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_MARGIN_INFINITE_SLAB = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_OK = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_PREC_FP64 = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_PREC_MIXED = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_PREC_MIXED_VISC = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_PROUGH_MARTIN2011 = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_PROUGH_MISMIPPLUS = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_PROUGH_SSA_ICESTREAM = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_RHEO_HUYBRECHTS1992 = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_RHEO_MISMIP_MOD = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_RHEO_UNIFORM = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ROUGH_PARAMETERISED = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ROUGH_PRESCRIBED = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_ROUGH_UNIFORM = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_COULOMB = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_COULOMB_REGULARISED = 3
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_IDEALISED = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_NO_SLIDING = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_SCHOOF2005 = 6
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_TSAI2015 = 5
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_WEERTMAN = 4
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SLID_ZOET_IVERSON = 7
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SOLVER_PETSC = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_SOLVER_SOR = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_STOP_PICARD = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_STOP_RESIDUAL = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TIME_OFF = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TIME_SMOOTHER = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TIME_VISC = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_CALVINGFRONT = 8
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_COAST = 5
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_GROUNDINGLINE = 7
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_LAKE = 2
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_LAND = 0
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_MARGIN = 6
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_OCEAN = 1
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_SHEET = 3
  INTEGER(C_INT32_T), PARAMETER :: IMAU_TYPE_SHELF = 4
  INTEGER(C_INT32_T), PARAMETER :: IMAU_NZ_MAX = 32

  TYPE, BIND(C) :: imau_grid
    INTEGER(C_INT32_T)   :: nx
    INTEGER(C_INT32_T)   :: ny
    REAL(C_DOUBLE)       :: dx
    TYPE(C_PTR)          :: x
    TYPE(C_PTR)          :: y
  END TYPE imau_grid

  TYPE, BIND(C) :: imau_cfg
    INTEGER(C_INT32_T)   :: choice_ice_dynamics
    INTEGER(C_INT32_T)   :: choice_ice_margin
    INTEGER(C_INT32_T)   :: choice_sliding_law
    INTEGER(C_INT32_T)   :: choice_idealised_sliding_law
    INTEGER(C_INT32_T)   :: choice_basal_hydrology
    INTEGER(C_INT32_T)   :: choice_basal_roughness
    INTEGER(C_INT32_T)   :: choice_param_basal_roughness
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_u_west
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_u_east
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_u_south
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_u_north
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_v_west
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_v_east
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_v_south
    INTEGER(C_INT32_T)   :: DIVA_boundary_BC_v_north
    INTEGER(C_INT32_T)   :: DIVA_choice_matrix_solver
    INTEGER(C_INT32_T)   :: include_SSADIVA_crossterms
    INTEGER(C_INT32_T)   :: do_GL_subgrid_friction
    INTEGER(C_INT32_T)   :: include_basal_freezing
    INTEGER(C_INT32_T)   :: nz
    REAL(C_DOUBLE)       :: zeta(32)
    REAL(C_DOUBLE)       :: n_flow
    REAL(C_DOUBLE)       :: DIVA_visc_it_norm_dUV_tol
    INTEGER(C_INT32_T)   :: DIVA_visc_it_nit
    REAL(C_DOUBLE)       :: DIVA_visc_it_relax
    REAL(C_DOUBLE)       :: DIVA_epsilon_sq_0
    REAL(C_DOUBLE)       :: DIVA_visc_eff_min
    REAL(C_DOUBLE)       :: DIVA_beta_max
    REAL(C_DOUBLE)       :: DIVA_vel_max
    REAL(C_DOUBLE)       :: slid_delta_v
    REAL(C_DOUBLE)       :: slid_Weertman_m
    REAL(C_DOUBLE)       :: slid_Coulomb_reg_q_plastic
    REAL(C_DOUBLE)       :: slid_Coulomb_reg_u_threshold
    REAL(C_DOUBLE)       :: slid_ZI_ut
    REAL(C_DOUBLE)       :: slid_ZI_p
    REAL(C_DOUBLE)       :: deltaT_basal_freezing
    REAL(C_DOUBLE)       :: Martin2011_hydro_Hb_min
    REAL(C_DOUBLE)       :: Martin2011_hydro_Hb_max
    REAL(C_DOUBLE)       :: Martin2011till_phi_Hb_min
    REAL(C_DOUBLE)       :: Martin2011till_phi_Hb_max
    REAL(C_DOUBLE)       :: Martin2011till_phi_min
    REAL(C_DOUBLE)       :: Martin2011till_phi_max
    REAL(C_DOUBLE)       :: SSA_icestream_L
    REAL(C_DOUBLE)       :: SSA_icestream_m
    REAL(C_DOUBLE)       :: ISMIP_HOM_L
    INTEGER(C_INT32_T)   :: precision
    INTEGER(C_INT32_T)   :: stop_rule
    REAL(C_DOUBLE)       :: nonlinear_rtol
    INTEGER(C_INT32_T)   :: mg_levels
    INTEGER(C_INT32_T)   :: check_interval
    REAL(C_DOUBLE)       :: picard_relax_max
    INTEGER(C_INT32_T)   :: mg_smoother
    INTEGER(C_INT32_T)   :: ksp_type
    INTEGER(C_INT32_T)   :: mg_rebuild
    INTEGER(C_INT32_T)   :: anderson_m
    INTEGER(C_INT32_T)   :: warm_visc_iters
    REAL(C_DOUBLE)       :: anderson_beta
    REAL(C_DOUBLE)       :: anderson_restart
    INTEGER(C_INT32_T)   :: warm_column_iters
    INTEGER(C_INT32_T)   :: stall_window
    REAL(C_DOUBLE)       :: stall_drop
    REAL(C_DOUBLE)       :: stall_relax
    INTEGER(C_INT32_T)   :: mg_graph
  END TYPE imau_cfg

  TYPE, BIND(C) :: imau_ice_io
    TYPE(C_PTR)          :: Hi_a
    TYPE(C_PTR)          :: Hb_a
    TYPE(C_PTR)          :: SL_a
    TYPE(C_PTR)          :: Hs_a
    TYPE(C_PTR)          :: TAF_a
    TYPE(C_PTR)          :: dHs_dx_a
    TYPE(C_PTR)          :: dHs_dy_a
    TYPE(C_PTR)          :: dHi_dx_a
    TYPE(C_PTR)          :: dHi_dy_a
    TYPE(C_PTR)          :: dHb_dt_a
    TYPE(C_PTR)          :: A_flow_vav_a
    TYPE(C_PTR)          :: mask_land_a
    TYPE(C_PTR)          :: mask_ocean_a
    TYPE(C_PTR)          :: mask_ice_a
    TYPE(C_PTR)          :: mask_sheet_a
    TYPE(C_PTR)          :: mask_shelf_a
    TYPE(C_PTR)          :: Hi_cx
    TYPE(C_PTR)          :: dHs_dx_cx
    TYPE(C_PTR)          :: dHs_dy_cx
    TYPE(C_PTR)          :: Hi_cy
    TYPE(C_PTR)          :: dHs_dx_cy
    TYPE(C_PTR)          :: dHs_dy_cy
    TYPE(C_PTR)          :: Hi_b
    TYPE(C_PTR)          :: A_flow_3D_a
    TYPE(C_PTR)          :: A_flow_3D_cx
    TYPE(C_PTR)          :: A_flow_3D_cy
    TYPE(C_PTR)          :: Ti_a
    TYPE(C_PTR)          :: Ti_pmp_a
    TYPE(C_PTR)          :: ISMIP_HOM_E_slides
    TYPE(C_PTR)          :: beta_sq_a
    TYPE(C_PTR)          :: alpha_sq_a
    TYPE(C_PTR)          :: phi_fric_a
    TYPE(C_PTR)          :: tauc_a
    TYPE(C_PTR)          :: u_vav_cx
    TYPE(C_PTR)          :: v_vav_cy
    TYPE(C_PTR)          :: u_SSA_cx
    TYPE(C_PTR)          :: v_SSA_cy
    TYPE(C_PTR)          :: taub_cx
    TYPE(C_PTR)          :: taub_cy
    TYPE(C_PTR)          :: visc_eff_3D_a
    TYPE(C_PTR)          :: u_3D_cx
    TYPE(C_PTR)          :: v_3D_cy
    TYPE(C_PTR)          :: u_3D_SIA_cx
    TYPE(C_PTR)          :: v_3D_SIA_cy
    TYPE(C_PTR)          :: u_3D_a
    TYPE(C_PTR)          :: v_3D_a
    TYPE(C_PTR)          :: w_3D_a
    TYPE(C_PTR)          :: F1_3D_a
    TYPE(C_PTR)          :: du_dz_3D_cx
    TYPE(C_PTR)          :: dv_dz_3D_cy
    TYPE(C_PTR)          :: u_vav_a
    TYPE(C_PTR)          :: v_vav_a
    TYPE(C_PTR)          :: u_surf_a
    TYPE(C_PTR)          :: v_surf_a
    TYPE(C_PTR)          :: u_base_a
    TYPE(C_PTR)          :: v_base_a
    TYPE(C_PTR)          :: uabs_vav_a
    TYPE(C_PTR)          :: uabs_surf_a
    TYPE(C_PTR)          :: uabs_base_a
    TYPE(C_PTR)          :: w_surf_a
    TYPE(C_PTR)          :: w_base_a
    TYPE(C_PTR)          :: R_shear
    TYPE(C_PTR)          :: u_surf_cx
    TYPE(C_PTR)          :: v_surf_cy
    TYPE(C_PTR)          :: u_base_cx
    TYPE(C_PTR)          :: v_base_cy
    TYPE(C_PTR)          :: beta_a
    TYPE(C_PTR)          :: beta_eff_a
    TYPE(C_PTR)          :: beta_eff_cx
    TYPE(C_PTR)          :: beta_eff_cy
    TYPE(C_PTR)          :: taudx_cx
    TYPE(C_PTR)          :: taudy_cy
    TYPE(C_PTR)          :: N_a
    TYPE(C_PTR)          :: N_b
    TYPE(C_PTR)          :: N_cx
    TYPE(C_PTR)          :: N_cy
    TYPE(C_PTR)          :: visc_eff_int_a
    TYPE(C_PTR)          :: F2_a
    TYPE(C_PTR)          :: f_grnd_a
    TYPE(C_PTR)          :: f_grnd_cx
    TYPE(C_PTR)          :: f_grnd_cy
    TYPE(C_PTR)          :: f_grnd_b
    TYPE(C_PTR)          :: overburden_pressure_a
    TYPE(C_PTR)          :: pore_water_pressure_a
    TYPE(C_PTR)          :: Neff_a
    TYPE(C_PTR)          :: DIVA_mask_combi
    TYPE(C_PTR)          :: DIVA_isfront_inner
    TYPE(C_PTR)          :: DIVA_isfront_outer
    TYPE(C_PTR)          :: u_cx_prev
    TYPE(C_PTR)          :: v_cy_prev
    TYPE(C_PTR)          :: DIVA_err_cx
    TYPE(C_PTR)          :: DIVA_err_cy
    INTEGER(C_INT32_T)   :: DIVA_SOR_nit
    REAL(C_DOUBLE)       :: DIVA_SOR_tol
    REAL(C_DOUBLE)       :: DIVA_SOR_omega
    REAL(C_DOUBLE)       :: DIVA_PETSc_rtol
    REAL(C_DOUBLE)       :: DIVA_PETSc_abstol
    INTEGER(C_INT32_T)   :: stat_picard_iterations
    INTEGER(C_INT64_T)   :: stat_linear_sweeps
    REAL(C_DOUBLE)       :: stat_resid_UV
    REAL(C_DOUBLE)       :: stat_nonlinear_residual
    REAL(C_DOUBLE)       :: stat_seconds
  END TYPE imau_ice_io

  TYPE, BIND(C) :: imau_thickness_cfg
    INTEGER(C_INT32_T)   :: choice_ice_integration_method
    INTEGER(C_INT32_T)   :: choice_ice_dynamics
    INTEGER(C_INT32_T)   :: ice_thickness_west_BC
    INTEGER(C_INT32_T)   :: ice_thickness_east_BC
    INTEGER(C_INT32_T)   :: ice_thickness_south_BC
    INTEGER(C_INT32_T)   :: ice_thickness_north_BC
    INTEGER(C_INT32_T)   :: dHi_choice_matrix_solver
    INTEGER(C_INT32_T)   :: dHi_SOR_nit
    REAL(C_DOUBLE)       :: dHi_SOR_tol
    REAL(C_DOUBLE)       :: dHi_SOR_omega
    REAL(C_DOUBLE)       :: dHi_PETSc_rtol
    REAL(C_DOUBLE)       :: dHi_PETSc_abstol
    REAL(C_DOUBLE)       :: dt_max
  END TYPE imau_thickness_cfg

  TYPE, BIND(C) :: imau_producer_cfg
    INTEGER(C_INT32_T)   :: nz
    REAL(C_DOUBLE)       :: zeta(32)
    INTEGER(C_INT32_T)   :: choice_ice_margin
    INTEGER(C_INT32_T)   :: do_ocean_floodfill
    INTEGER(C_INT32_T)   :: choice_ice_rheology
    REAL(C_DOUBLE)       :: uniform_flow_factor
    REAL(C_DOUBLE)       :: m_enh_sheet
    REAL(C_DOUBLE)       :: m_enh_shelf
  END TYPE imau_producer_cfg

  TYPE, BIND(C) :: imau_timestep_cfg
    REAL(C_DOUBLE)       :: start_time_of_run
    REAL(C_DOUBLE)       :: end_time_of_run
    REAL(C_DOUBLE)       :: dt_min
    REAL(C_DOUBLE)       :: dt_max
    REAL(C_DOUBLE)       :: dt_startup_phase
    INTEGER(C_INT32_T)   :: choice_calving_law
    INTEGER(C_INT32_T)   :: fixed_shelf_geometry
    INTEGER(C_INT32_T)   :: fixed_sheet_geometry
    INTEGER(C_INT32_T)   :: fixed_grounding_line
    INTEGER(C_INT32_T)   :: do_remove_shelves
    INTEGER(C_INT32_T)   :: remove_shelves_larger_than_PD
    INTEGER(C_INT32_T)   :: continental_shelf_calving
    INTEGER(C_INT32_T)   :: pad0_
    REAL(C_DOUBLE)       :: calving_threshold_thickness
    REAL(C_DOUBLE)       :: continental_shelf_min_height
    REAL(C_DOUBLE)       :: pc_epsilon
    REAL(C_DOUBLE)       :: pc_k_I
    REAL(C_DOUBLE)       :: pc_k_p
    REAL(C_DOUBLE)       :: pc_eta_min
  END TYPE imau_timestep_cfg

  TYPE, BIND(C) :: imau_refgeo_io
    TYPE(C_PTR)          :: mask_noice_a
    TYPE(C_PTR)          :: Hi_PD
    TYPE(C_PTR)          :: Hb_PD
    TYPE(C_PTR)          :: Hi_GIAeq
    TYPE(C_PTR)          :: Hb_GIAeq
  END TYPE imau_refgeo_io

  TYPE, BIND(C) :: imau_producer_io
    TYPE(C_PTR)          :: Hi_a
    TYPE(C_PTR)          :: Hb_a
    TYPE(C_PTR)          :: SL_a
    TYPE(C_PTR)          :: dHi_dt_a
    TYPE(C_PTR)          :: dHb_dt_a
    TYPE(C_PTR)          :: Ti_a
    TYPE(C_PTR)          :: Hs_a
    TYPE(C_PTR)          :: TAF_a
    TYPE(C_PTR)          :: dHs_dt_a
    TYPE(C_PTR)          :: mask_land_a
    TYPE(C_PTR)          :: mask_ocean_a
    TYPE(C_PTR)          :: mask_ice_a
    TYPE(C_PTR)          :: mask_sheet_a
    TYPE(C_PTR)          :: mask_shelf_a
    TYPE(C_PTR)          :: mask_coast_a
    TYPE(C_PTR)          :: mask_margin_a
    TYPE(C_PTR)          :: mask_gl_a
    TYPE(C_PTR)          :: mask_cf_a
    TYPE(C_PTR)          :: mask_a
    TYPE(C_PTR)          :: Hi_cx
    TYPE(C_PTR)          :: Hi_cy
    TYPE(C_PTR)          :: Hi_b
    TYPE(C_PTR)          :: A_flow_3D_a
    TYPE(C_PTR)          :: A_flow_vav_a
    TYPE(C_PTR)          :: A_flow_3D_cx
    TYPE(C_PTR)          :: A_flow_3D_cy
    TYPE(C_PTR)          :: A_flow_vav_cx
    TYPE(C_PTR)          :: A_flow_vav_cy
    TYPE(C_PTR)          :: dHi_dx_a
    TYPE(C_PTR)          :: dHi_dy_a
    TYPE(C_PTR)          :: dHs_dx_a
    TYPE(C_PTR)          :: dHs_dy_a
    TYPE(C_PTR)          :: dHs_dx_cx
    TYPE(C_PTR)          :: dHs_dy_cx
    TYPE(C_PTR)          :: dHs_dx_cy
    TYPE(C_PTR)          :: dHs_dy_cy
    TYPE(C_PTR)          :: float_margin_frac_a
    TYPE(C_PTR)          :: Hi_eff_cf_a
  END TYPE imau_producer_io

  TYPE, BIND(C) :: imau_timestep_state
    REAL(C_DOUBLE)       :: time
    REAL(C_DOUBLE)       :: t_next_SIA
    REAL(C_DOUBLE)       :: t_next_SSA
    REAL(C_DOUBLE)       :: dt_crit_SIA
    REAL(C_DOUBLE)       :: dt_crit_SSA
    REAL(C_DOUBLE)       :: dt
    INTEGER(C_INT32_T)   :: nsteps
  END TYPE imau_timestep_state

  TYPE, BIND(C) :: imau_pc_state
    REAL(C_DOUBLE)       :: pc_zeta
    REAL(C_DOUBLE)       :: pc_eta
    REAL(C_DOUBLE)       :: pc_eta_prev
    REAL(C_DOUBLE)       :: dt_crit_ice
    REAL(C_DOUBLE)       :: dt_crit_ice_prev
    REAL(C_DOUBLE)       :: dt
    REAL(C_DOUBLE)       :: t_next
    TYPE(C_PTR)          :: dHidt_Hn_un
    TYPE(C_PTR)          :: dHi_dt_a
  END TYPE imau_pc_state

  INTERFACE
    FUNCTION imau_vel_init(grid, cfg, ctx) BIND(C, name='imau_vel_init') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg
      TYPE(imau_grid), INTENT(IN) :: grid
      TYPE(imau_cfg),  INTENT(IN) :: cfg
      TYPE(C_PTR),     INTENT(OUT) :: ctx
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_solve_diva(ctx, grid, cfg, io) BIND(C, name='imau_vel_solve_diva') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg, imau_ice_io
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),   INTENT(IN)    :: grid
      TYPE(imau_cfg),    INTENT(IN)    :: cfg
      TYPE(imau_ice_io), INTENT(INOUT) :: io
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_solve_ssa(ctx, grid, cfg, io) BIND(C, name='imau_vel_solve_ssa') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg, imau_ice_io
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),   INTENT(IN)    :: grid
      TYPE(imau_cfg),    INTENT(IN)    :: cfg
      TYPE(imau_ice_io), INTENT(INOUT) :: io
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_solve_sia(ctx, grid, cfg, io) BIND(C, name='imau_vel_solve_sia') RESULT(rc)
      IMPORT :: C_INT, C_PTR, imau_grid, imau_cfg, imau_ice_io
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),   INTENT(IN)    :: grid
      TYPE(imau_cfg),    INTENT(IN)    :: cfg
      TYPE(imau_ice_io), INTENT(INOUT) :: io
      INTEGER(C_INT) :: rc
    END FUNCTION
    SUBROUTINE imau_vel_finalize(ctx) BIND(C, name='imau_vel_finalize')
      IMPORT :: C_PTR
      TYPE(C_PTR), VALUE :: ctx
    END SUBROUTINE
    FUNCTION imau_vel_keep_memory(ctx, bytes, kept) BIND(C, name='imau_vel_keep_memory') RESULT(rc)
      IMPORT :: C_INT, C_INT64_T, C_PTR
      TYPE(C_PTR), VALUE :: ctx
      INTEGER(C_INT64_T), VALUE :: bytes
      INTEGER(C_INT64_T), INTENT(OUT) :: kept
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_vel_last_error(ctx) BIND(C, name='imau_vel_last_error') RESULT(msg)
      IMPORT :: C_PTR
      TYPE(C_PTR), VALUE :: ctx
      TYPE(C_PTR) :: msg
    END FUNCTION
    SUBROUTINE imau_vel_default_config(cfg) BIND(C, name='imau_vel_default_config')
      IMPORT :: imau_cfg
      TYPE(imau_cfg), INTENT(OUT) :: cfg
    END SUBROUTINE
    ! run_ice_dynamics_direct / _pc with update_ice_thickness (ref, geo: C_LOC or C_NULL_PTR)
    FUNCTION imau_run_ice_dynamics_direct(ctx, grid, cfg, tcfg, pcfg, scfg, io, ref, SMB_year, BMB, Hi_end, &
                                          geo, st, t_end) BIND(C, name='imau_run_ice_dynamics_direct') RESULT(rc)
      IMPORT :: C_INT, C_PTR, C_DOUBLE, imau_grid, imau_cfg, imau_thickness_cfg, imau_producer_cfg, &
                imau_timestep_cfg, imau_ice_io, imau_timestep_state
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),           INTENT(IN)    :: grid
      TYPE(imau_cfg),            INTENT(IN)    :: cfg
      TYPE(imau_thickness_cfg),  INTENT(IN)    :: tcfg
      TYPE(imau_producer_cfg),   INTENT(IN)    :: pcfg
      TYPE(imau_timestep_cfg),   INTENT(IN)    :: scfg
      TYPE(imau_ice_io),         INTENT(INOUT) :: io
      TYPE(C_PTR), VALUE :: ref
      REAL(C_DOUBLE),            INTENT(IN)    :: SMB_year(*), BMB(*)
      REAL(C_DOUBLE),            INTENT(OUT)   :: Hi_end(*)
      TYPE(C_PTR), VALUE :: geo
      TYPE(imau_timestep_state), INTENT(INOUT) :: st
      REAL(C_DOUBLE), VALUE :: t_end
      INTEGER(C_INT) :: rc
    END FUNCTION
    FUNCTION imau_run_ice_dynamics_pc(ctx, grid, cfg, tcfg, pcfg, scfg, io, ref, SMB_year, BMB, Hi_end, &
                                      geo, st, pc, t_end) BIND(C, name='imau_run_ice_dynamics_pc') RESULT(rc)
      IMPORT :: C_INT, C_PTR, C_DOUBLE, imau_grid, imau_cfg, imau_thickness_cfg, imau_producer_cfg, &
                imau_timestep_cfg, imau_ice_io, imau_timestep_state, imau_pc_state
      TYPE(C_PTR), VALUE :: ctx
      TYPE(imau_grid),           INTENT(IN)    :: grid
      TYPE(imau_cfg),            INTENT(IN)    :: cfg
      TYPE(imau_thickness_cfg),  INTENT(IN)    :: tcfg
      TYPE(imau_producer_cfg),   INTENT(IN)    :: pcfg
      TYPE(imau_timestep_cfg),   INTENT(IN)    :: scfg
      TYPE(imau_ice_io),         INTENT(INOUT) :: io
      TYPE(C_PTR), VALUE :: ref
      REAL(C_DOUBLE),            INTENT(IN)    :: SMB_year(*), BMB(*)
      REAL(C_DOUBLE),            INTENT(OUT)   :: Hi_end(*)
      TYPE(C_PTR), VALUE :: geo
      TYPE(imau_timestep_state), INTENT(INOUT) :: st
      TYPE(imau_pc_state),       INTENT(INOUT) :: pc
      REAL(C_DOUBLE), VALUE :: t_end
      INTEGER(C_INT) :: rc
    END FUNCTION
  END INTERFACE

CONTAINS

  ! copy the C error string of a context into a Fortran string
  FUNCTION imau_vel_error_text(ctx) RESULT(txt)
    TYPE(C_PTR), INTENT(IN) :: ctx
    CHARACTER(LEN=512) :: txt
    CHARACTER(KIND=C_CHAR), DIMENSION(:), POINTER :: p
    INTEGER :: k
    TYPE(C_PTR) :: cp
    INTERFACE
      FUNCTION strlen(s) BIND(C, name='strlen') RESULT(n)
        IMPORT :: C_PTR, C_SIZE_T
        TYPE(C_PTR), VALUE :: s
        INTEGER(C_SIZE_T) :: n
      END FUNCTION
    END INTERFACE
    txt = ' '
    cp = imau_vel_last_error(ctx)
    IF (.NOT. C_ASSOCIATED(cp)) RETURN
    CALL C_F_POINTER(cp, p, [INT(strlen(cp))])
    DO k = 1, MIN(SIZE(p), LEN(txt))
      txt(k:k) = p(k)
    END DO
  END FUNCTION imau_vel_error_text

END MODULE imau_vel_bindings
